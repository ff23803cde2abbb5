"""The work a user of boltmi has it do, as cases that can be timed one by one.

A case is a dict of plain values; `kind` names the entry point.  Sizes follow
the repository's own uses: Bolt's test and example settings (100 k, ℓᵧ = 8,
reltol 1e-11; plin's defaults), the full CMB spectrum of bench.py (800 k,
ℓᵧ = ℓ_ν = 50, ℓ ≤ 2500 on 5000 dense k), batches over cosmologies, and the
Bessel moments of src/bessel.  Cosmologies are drawn from a parameter box around
Bolt's default, so that every state has tables of its own.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "bolt.jl_amd"))
import boltmi  # noqa: E402
from boltmi import _abi  # noqa: E402

NX, X0, X1 = 2001, -20.0, 0.0  # the x grid every table and source grid has
NXI = 799                      # of these, the left-sum nodes after x = -8


def listed():
    return [
        # one wavenumber of the linear power spectrum with plin's defaults (n = 473): the smallest solver call, as in
        # a root search for k_nl or a plot's single point; one mode's latency and the launch
        dict(name="plin_one", kind="plin", nk=1, kmin=0.05, kmax=0.05, lg=50, ln=50, lm=20, x=0.0, reltol=1e-5),
        # a P(k) table: 200 log-spaced k, plin's defaults, what a likelihood asks for per cosmology
        dict(name="plin_200", kind="plin", nk=200, kmin=1e-4, kmax=0.5, lg=50, ln=50, lm=20, x=0.0, reltol=1e-5),
        # boltsolve of one Hierarchy at Bolt's defaults, the solution on the whole x grid, as the reference's tests
        # and notebooks look at a mode
        dict(name="boltsolve_one", kind="boltsolve", nk=1, kmin=0.03, kmax=0.03, l=8, reltol=1e-6, nsave=2001),
        # source_grid as Bolt's test suite calls it: 100 quadratic k, ℓᵧ = 8
        dict(name="source_100", kind="source", nk=100, kmin=7e-5, kmax=0.3, lg=8, ln=8, lm=10, reltol=1e-11),
        # both sources for a few cosmologies in one launch (a parameter scan's inner call), odd k count
        dict(name="source_batch", kind="batch", nc=5, nk=77, kmin=1e-4, kmax=0.2, lg=20, ln=20, lm=10, reltol=1e-11),
        # the whole CMB spectrum, device resident: source_grid of 800 k, then C_ℓ^TT for every ℓ ≤ 2500
        dict(name="spectrum_800", kind="spectrum", nk=800, kmin=1e-4, kmax=0.5, lg=50, lmax=2500, lstep=1, nkd=5000),
        # C_ℓ^TT from a source grid the user holds on the host, every tenth ℓ as in the CAMB comparison of Bolt's tests
        dict(name="cltt_250", kind="cl", nk=100, kmax=0.3, lmin=10, lmax=2500, lstep=10, nkd=5000, pol=False, mode=0),
        # TT, TE and EE together for every ℓ ≤ 1500
        dict(name="cl_ttteee", kind="cl", nk=200, kmax=0.35, lmin=2, lmax=1500, lstep=1, nkd=3001, pol=True, mode=0),
        # Bolt's own discretisation of j_ℓ (5001-node splines), its test's ℓ list
        dict(name="cltt_spline", kind="cl", nk=100, kmax=0.3, lmin=10, lmax=1200, lstep=10, nkd=5000, pol=False, mode=1),
        # dC_ℓ/dp of a spectrum by forward-mode Duals: the tangent solve and the tangent line-of-sight sum
        dict(name="jvp_spectrum", kind="jvp", nk=60, kmin=1e-4, kmax=0.15, lg=8, lmax=600, lstep=1, nkd=1000),
        # a Bessel moment table and the Filon rule on it for many wavenumbers
        dict(name="filon", kind="filon", nu=2, order=3, nodes=400_000, xmax=2000.0, nt=1001, nk=700),
        # background and recombination tables of a batch of cosmologies on the GPU
        dict(name="tables_96", kind="tables", nc=96),
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def draw(rng):
    kind = rng.choice(["plin", "plin", "boltsolve", "source", "source", "batch", "spectrum", "cl", "cl", "cl", "jvp",
                       "filon", "tables"])
    if kind == "plin":
        nk = round(_log(rng, 1, 200))
        kmax = _log(rng, 2e-3, 0.5)
        lg = rng.randint(8, 50)
        return dict(kind=kind, nk=nk, kmin=kmax if nk == 1 else kmax * _log(rng, 1e-3, 0.3), kmax=kmax, lg=lg, ln=lg,
                    lm=rng.randint(8, 20), x=rng.choice([0.0, 0.0, -1.0, -2.5]), reltol=10 ** rng.uniform(-7, -4))
    if kind == "boltsolve":
        nk = rng.randint(1, 6)
        kmax = _log(rng, 2e-3, 0.2)
        return dict(kind=kind, nk=nk, kmin=kmax if nk == 1 else kmax * _log(rng, 1e-2, 0.5), kmax=kmax,
                    l=rng.randint(6, 30), reltol=10 ** rng.uniform(-9, -5), nsave=rng.choice([1, 50, 401, 1001, 2001]))
    if kind == "source":
        lg = rng.randint(6, 50)
        return dict(kind=kind, nk=round(_log(rng, 5, 800)), kmin=_log(rng, 5e-5, 1e-3), kmax=_log(rng, 0.02, 0.5),
                    lg=lg, ln=rng.choice([8, lg]), lm=rng.randint(8, 14), reltol=rng.choice([1e-11, 1e-9, 1e-7]))
    if kind == "batch":
        lg = rng.randint(8, 50)
        return dict(kind=kind, nc=rng.randint(2, 8), nk=round(_log(rng, 10, 200)), kmin=1e-4,
                    kmax=_log(rng, 0.03, 0.4), lg=lg, ln=lg, lm=10, reltol=1e-11)
    if kind == "spectrum":
        return dict(kind=kind, nk=round(_log(rng, 50, 800)), kmin=1e-4, kmax=_log(rng, 0.05, 0.5),
                    lg=rng.randint(8, 50), lmax=round(_log(rng, 100, 2500)), lstep=1, nkd=round(_log(rng, 300, 5000)))
    if kind == "cl":
        return dict(kind=kind, nk=round(_log(rng, 30, 800)), kmax=_log(rng, 0.05, 0.5), lmin=rng.choice([2, 2, 10]),
                    lmax=round(_log(rng, 50, 2500)), lstep=rng.choice([1, 1, 3, 10]), nkd=round(_log(rng, 200, 5000)),
                    pol=rng.random() < 0.4, mode=0 if rng.random() < 0.75 else 1)
    if kind == "jvp":
        return dict(kind=kind, nk=round(_log(rng, 10, 200)), kmin=1e-4, kmax=_log(rng, 0.03, 0.3),
                    lg=rng.randint(6, 50), lmax=round(_log(rng, 100, 1500)), lstep=rng.choice([1, 7]),
                    nkd=round(_log(rng, 200, 3000)))
    if kind == "filon":
        return dict(kind=kind, nu=rng.choice([2, 3]), order=rng.choice([3, 4]), nodes=round(_log(rng, 2e4, 2e6)),
                    xmax=_log(rng, 300.0, 5000.0), nt=round(_log(rng, 100, 2500)), nk=round(_log(rng, 10, 2000)))
    return dict(kind="tables", nc=round(_log(rng, 1, 96)))


# ------------------------------------------------------------------- inputs
def _cosmology(r):
    """a cosmology of the box; a third of them with massless neutrinos"""
    mnu = 0.0 if r.random() < 0.33 else r.uniform(0.02, 0.3) * boltmi.MASS_NATURAL
    return boltmi.CosmoParams(h=r.uniform(0.62, 0.76), Ω_b=r.uniform(0.042, 0.052), Ω_c=r.uniform(0.2, 0.27),
                              A=r.uniform(1.9e-9, 2.3e-9), n=r.uniform(0.93, 1.0), Y_p=r.uniform(0.235, 0.255),
                              Σm_ν=mnu)


def _tables(par):
    bg = boltmi.Background(par)
    return par, bg, boltmi.IonizationHistory(boltmi.RECFAST(bg), par, bg)


def _kgrid(case, r):
    """log-spaced k, its ends moved by up to a percent from seed to seed"""
    s = 1.0 + 0.01 * r.uniform(-1, 1)
    if case["nk"] == 1:
        return np.array([case["kmax"] * s])
    return np.logspace(math.log10(case["kmin"] * s), math.log10(case["kmax"] * s), case["nk"])


def _ells(case):
    return np.arange(case.get("lmin", 2), case["lmax"] + 1, case["lstep"], dtype=np.int32)


def _sources(case, r, bg):
    """source grids of the shape the solver gives: the visibility peak with acoustic oscillations and damping in k,
    reionization, a late-time tail; the polarization source carries its 1/y²"""
    x = np.array([(X0 * (NX - 1 - j) + X1 * j) / (NX - 1) for j in range(NX)])
    k = np.logspace(-4, math.log10(case["kmax"]), case["nk"])[:, None]
    rs, amp, ph = 140.0 * r.uniform(0.9, 1.1), r.uniform(0.8, 1.2, 4), r.uniform(0, 0.5)
    g = np.exp(-0.5 * ((x + 7.0) / 0.07) ** 2) * 5.0 + np.exp(-0.5 * ((x + 2.2) / 0.25) ** 2) * 0.15
    damp = np.exp(-(k / 0.14) ** 2)
    S = g * (amp[0] * 0.2 + amp[1] * 0.4 * np.cos(k * rs + ph)) * damp
    S = S + amp[2] * 0.1 * np.exp(-0.5 * (x / 0.7) ** 2) / (1 + (k / 0.01) ** 2)
    y = k * (bg.eta0 - bg.eta(x))
    with np.errstate(divide="ignore"):
        P = 0.75 * g * amp[3] * 0.05 * np.sin(k * rs + ph) * damp / (y * y)
    return np.ascontiguousarray(S), np.ascontiguousarray(P)


def prepare(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    kind = case["kind"]
    if kind == "filon":
        # the piecewise quadratic of a smooth kernel on a time grid, wavenumbers with k t inside and past the table
        t = np.sort(r.uniform(0.0, 100.0, case["nt"]))
        t[0] = 0.0
        a, b = r.uniform(0.5, 1.5), r.uniform(0.02, 0.06)
        f = a * np.exp(-b * t) * np.cos(0.3 * t)
        fp = a * np.exp(-b * t) * (-b * np.cos(0.3 * t) - 0.3 * np.sin(0.3 * t))
        fpp = a * np.exp(-b * t) * ((b * b - 0.09) * np.cos(0.3 * t) + 0.6 * b * np.sin(0.3 * t))
        ks = np.sort(np.exp(r.uniform(math.log(0.05), math.log(1.1 * case["xmax"] / 100.0), case["nk"])))
        return dict(case=case, t=t, f=f, fp=fp, fpp=fpp, k=ks)
    if kind == "tables":
        return dict(case=case, pars=[_cosmology(r) for _ in range(case["nc"])])
    if kind == "batch":
        cosmos = boltmi.backgrounds([_cosmology(r) for _ in range(case["nc"])])
        return dict(case=case, cosmos=cosmos, k=_kgrid(case, r))
    par = _cosmology(r)
    if kind == "jvp":
        # ∂/∂Ω_b, as examples/plot_deriv_cl.jl differentiates
        par = boltmi.CosmoParams(h=par.h, Ω_b=boltmi.Dual(par.Ω_b, 1.0), Ω_c=par.Ω_c, A=par.A, n=par.n, Y_p=par.Y_p,
                                 Σm_ν=par.Σm_ν)
    par, bg, ih = _tables(par)
    st = dict(case=case, par=par, bg=bg, ih=ih)
    H0 = float(boltmi.dual.value(bg.H0))
    if kind == "cl":
        S, P = _sources(case, r, bg)
        ks = np.logspace(-4, math.log10(case["kmax"]), case["nk"])
        st.update(S=boltmi.SourceGrid(bg.x_grid, ks, S), P=boltmi.SourceGrid(bg.x_grid, ks, P), ells=_ells(case),
                  dense=boltmi.quadratic_k(0.01 * H0, 1000 * H0, case["nkd"]))
        return st
    st["k"] = _kgrid(case, r)
    if kind == "boltsolve":
        st["x"] = bg.x_grid if case["nsave"] == NX else np.linspace(-12.0, 0.0, case["nsave"]) if case["nsave"] > 1 \
            else np.array([0.0])
    if kind in ("spectrum", "jvp"):
        st.update(ells=_ells(case), dense=boltmi.quadratic_k(0.01 * H0, 1000 * H0, case["nkd"]))
    if kind == "spectrum":
        dev = dict(dtype=torch.float64, device="cuda")
        st.update(ctx=boltmi.default_context(), cfg=boltmi.hier_cfg(case["lg"], case["lg"], 10, 15, 1e-11, 1e-6),
                  d_k=torch.tensor(st["k"], **dev), d_dense=torch.tensor(st["dense"], **dev),
                  d_S=torch.zeros((case["nk"], NX), **dev), d_cl=torch.zeros(len(st["ells"]), **dev),
                  d_status=torch.zeros(case["nk"], dtype=torch.int32, device="cuda"))
        st["cid"] = bg.cosmo_id(st["ctx"])
        torch.cuda.synchronize()
    return st


# --------------------------------------------------------------------- pass
def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "filon":
        itp = boltmi.sph_bessel_interpolator(case["nu"], case["order"], 0.0, case["xmax"], case["nodes"])
        out = boltmi.filon_sum(itp, st["t"], st["f"], st["fp"], st["fpp"], st["k"])
        itp.close()
        return out
    if kind == "tables":
        got = boltmi.backgrounds(st["pars"], device=True)
        return dict(coef=np.stack([b.coef for _, b, _ in got]), scal=np.stack([b.scal for _, b, _ in got]))
    if kind == "batch":
        T, P = boltmi.source_grid_batch(st["cosmos"], st["k"], ℓᵧ=case["lg"], ℓ_ν=case["ln"], ℓ_mν=case["lm"],
                                        reltol=case["reltol"], want_p=True)
        return dict(T=np.stack([s.grid for s in T]), P=np.stack([s.grid for s in P]))
    par, bg, ih = st["par"], st["bg"], st["ih"]
    if kind == "plin":
        k = st["k"] if case["nk"] > 1 else float(st["k"][0])
        return boltmi.plin(k, par, bg, ih, 15, case["lg"], case["ln"], case["lm"], case["x"], case["reltol"])
    if kind == "boltsolve":
        if case["nk"] == 1:
            h = boltmi.Hierarchy(boltmi.BasicNewtonian(), par, bg, ih, float(st["k"][0]), case["l"])
            return boltmi.boltsolve(h, reltol=case["reltol"], saveat=st["x"]).u
        cfg = boltmi.hier_cfg(case["l"], reltol=case["reltol"])
        return boltmi.boltsolve_batch(par, bg, cfg, st["k"], st["x"])[0]
    if kind == "source":
        return boltmi.source_grid(par, bg, ih, st["k"], boltmi.BasicNewtonian(), case["lg"], case["reltol"],
                                  ℓ_ν=case["ln"], ℓ_mν=case["lm"]).grid
    if kind == "spectrum":
        L, h = _abi.lib(), st["ctx"].handle
        _abi.check(L.bolt_source_grid_dev(h, st["cid"], ctypes.byref(st["cfg"]), _ptr(st["d_k"]), case["nk"],
                                          _ptr(st["d_S"]), _ptr(st["d_status"]), None, None))
        _abi.check(L.bolt_cltt_dev(h, st["cid"], _ptr(st["d_S"]), _ptr(st["d_k"]), case["nk"], _ptr(st["d_dense"]),
                                   case["nkd"], _abi.pi(st["ells"]), len(st["ells"]), _ptr(st["d_cl"]), None, None))
        return dict(S=st["d_S"], cl=st["d_cl"], status=st["d_status"])
    if kind == "jvp":
        sf = boltmi.source_grid(par, bg, ih, st["k"], boltmi.BasicNewtonian(), case["lg"])
        cl = boltmi.cltt_on_grid(st["ells"], sf, st["dense"], par, bg)
        return dict(S=sf.grid.v, dS=sf.grid.d, cl=cl.v, dcl=cl.d)
    if case["pol"]:
        tt, te, ee = boltmi.cl_on_grid(st["ells"], st["S"], st["P"], st["dense"], par, bg, case["mode"])
        return dict(tt=tt, te=te, ee=ee)
    return dict(tt=boltmi.cltt_on_grid(st["ells"], st["S"], st["dense"], par, bg, case["mode"]))


# --------------------------------------------------------------------- work
def _steps(ks):
    """KenCarp4 steps of these modes: a few hundred for the expansion, the rest resolves the oscillations in kη"""
    return float(np.sum(400.0 + 9000.0 * ks))


def _solve_flops(ks, n, nq=15):
    """FP64 operations of the structured solve: per step five stage right-hand sides, banded factors, four
    substitutions and the border, the error solve, and the derivative at the new point"""
    rhs = 16 * n + 4 * nq + 40
    stage = rhs + 56 * n + 4 * (4 * nq + 40)
    return _steps(ks) * (73 * n + 5 * stage + rhs)


def _nstate(lg, ln, lm, nq=15):
    return 2 * (lg + 1) + (ln + 1) + (lm + 1) * nq + 5


def _los_flops(case, nsrc):
    """four operations a term and source; a term beyond the turning point ℓ = k (η₀ − η) vanishes"""
    H0 = 0.7 / 2997.9
    kd = 0.01 * H0 + (1000 - 0.01) * H0 * (np.arange(1, case["nkd"]) / case["nkd"]) ** 2
    return 2.0 * (1 + nsrc) * NXI * float(np.sum(np.minimum(case["lmax"], kd * 1.3e4)))


def work(case):
    kind = case["kind"]
    tab = 8.0 * 16 * (NX + 2)  # one cosmology's coefficient tables
    if kind == "filon":
        return dict(bytes=8.0 * (4 * case["nt"] + 2 * case["nk"] + case["order"] * (case["nodes"] + 2)),
                    flops=case["nodes"] * case["order"] * 30.0 + case["nk"] * case["nt"] * (case["order"] * 12.0 + 20))
    if kind == "tables":
        # some 2e5 recombination rate evaluations a cosmology, a hundred operations each
        return dict(bytes=case["nc"] * tab, flops=case["nc"] * 2e5 * 100.0)
    if kind == "cl":
        nout = len(_ells(case)) * (3 if case["pol"] else 1)
        return dict(bytes=8.0 * (case["nk"] * NXI * (2 if case["pol"] else 1) + case["nkd"] + nout),
                    flops=_los_flops(case, 2 if case["pol"] else 1))
    ks = np.array([case["kmax"]]) if case["nk"] == 1 else \
        np.logspace(math.log10(case["kmin"]), math.log10(case["kmax"]), case["nk"])
    if kind == "plin":
        return dict(bytes=tab + 16.0 * case["nk"], flops=_solve_flops(ks, _nstate(case["lg"], case["ln"], case["lm"])))
    if kind == "boltsolve":
        n = _nstate(case["l"], 8, 10)
        return dict(bytes=tab + 8.0 * case["nk"] * case["nsave"] * n, flops=_solve_flops(ks, n))
    if kind == "source":
        return dict(bytes=tab + 8.0 * case["nk"] * NX, flops=_solve_flops(ks, _nstate(case["lg"], case["ln"], case["lm"])))
    if kind == "batch":
        return dict(bytes=case["nc"] * (tab + 16.0 * case["nk"] * NX),
                    flops=case["nc"] * _solve_flops(ks, _nstate(case["lg"], case["ln"], case["lm"])))
    if kind == "spectrum":
        return dict(bytes=tab + 8.0 * (case["nk"] * NX + len(_ells(case))),
                    flops=_solve_flops(ks, _nstate(case["lg"], case["lg"], 10)) + _los_flops(case, 1))
    # jvp: the value and one derivative
    return dict(bytes=2 * (tab + 8.0 * (case["nk"] * NX + len(_ells(case)))),
                flops=2 * (_solve_flops(ks, _nstate(case["lg"], 8, 10)) + _los_flops(case, 1)))


# -------------------------------------------------------------------- exact
def _bessel_sums(z, ells, weights):
    """Σ_x j_ℓ(z) w for each ℓ of the ascending list and each w: Miller's downward recurrence in 64 bits, twice (the
    first time for the normalisation).  z [nk, nx], w [nk, nx] -> [len(weights)][len(ells), nk]"""
    lmax = int(ells[-1])
    zm = max(float(lmax), float(z.max()))
    top = int(zm + 80 + 14 * zm ** (1 / 3))
    inv = 1.0 / z
    want = {int(l): i for i, l in enumerate(ells)}
    out = [torch.zeros((len(ells), z.shape[0]), dtype=z.dtype, device=z.device) for _ in weights]
    total = None
    for pas in range(2):
        fp, fc = torch.zeros_like(z), torch.full_like(z, 1e-300)
        cnt = torch.zeros_like(z)
        for l in range(top, 0, -1):
            fp, fc = fc, (2 * l + 1) * inv * fc - fp
            big = fc.abs() > 1e250
            s = torch.ones_like(z).masked_fill_(big, 1e-250)
            fp, fc, cnt = fp * s, fc * s, cnt + big
            i = want.get(l - 1) if pas else None
            if i is not None:
                left = total - cnt
                v = torch.where(left == 0, fc, torch.where(left == 1, fc * 1e-250, torch.zeros_like(fc))) * norm
                for o, w in zip(out, weights):
                    o[i] = (v * w).sum(1)
        if not pas:
            total = cnt
            j0 = torch.sin(z) / z
            j1 = (j0 - torch.cos(z)) / z
            j1 = torch.where(z < 0.05, z / 3 * (1 - z * z / 10 * (1 - z * z / 28 * (1 - z * z / 54))), j1)
            norm = torch.where(j0.abs() >= j1.abs(), j0 / fc, j1 / fp)
    return out


def _exact_cl(case, seed):
    st = prepare(case, seed)
    bg, par = st["bg"], st["par"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def T(a):
        return torch.tensor(np.asarray(a), dtype=torch.float64, device=dev)

    x = np.array([(X0 * (NX - 1 - j) + X1 * j) / (NX - 1) for j in range(NX)])
    i0 = int(np.nonzero(x > -8.0)[0][0])
    at = slice(i0, NX - 1)
    dx = T(np.diff(x)[i0:])
    deta = T(bg.eta0 - bg.eta(x[at]))
    dense = st["dense"]
    km, dk = (dense[1:] + dense[:-1]) / 2, np.diff(dense)
    ksrc = st["S"].k_grid
    ia = np.clip(np.searchsorted(ksrc, km, side="right") - 1, 0, len(ksrc) - 2)
    tt = T((km - ksrc[ia]) / (ksrc[ia + 1] - ksrc[ia]))[:, None]
    ia = torch.tensor(ia, device=dev)
    ws = []
    for g in (st["S"].grid, st["P"].grid)[: 2 if case["pol"] else 1]:
        g = T(g[:, at])
        ws.append(((1 - tt) * g[ia] + tt * g[ia + 1]) * dx)
    kk = T(km)
    sums = _bessel_sums(kk[:, None] * deta, st["ells"], ws)
    Pw = par.A * (kk / 0.05) ** (par.n - 1.0) * T(dk) / kk
    l = T(st["ells"].astype(np.float64))
    spin = torch.sqrt((l + 2) * (l + 1) * l * (l - 1))
    res = dict(tt=4 * math.pi * (sums[0] ** 2 * Pw).sum(1))
    if case["pol"]:
        res["te"] = 4 * math.pi * spin * (sums[0] * sums[1] * Pw).sum(1)
        res["ee"] = 4 * math.pi * spin ** 2 * (sums[1] ** 2 * Pw).sum(1)
    return res


def _exact_filon(case, seed):
    """Gauss-Legendre panels of the quadratic times j_ν, two radians of k t each"""
    st = prepare(case, seed)
    t, f, fp, fpp, ks = (st[k] for k in ("t", "f", "fp", "fpp", "k"))
    if case["nk"] * case["nt"] > 2_000_000 or ks[-1] * np.max(np.diff(t)) > 120.0:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    xg, wg = np.polynomial.legendre.leggauss(20)
    xg, wg = (torch.tensor(v, device=dev) for v in (xg, wg))
    a, b = (torch.tensor(v, device=dev) for v in (t[:-1], t[1:]))
    F, Fp, Fpp = (torch.tensor(v[:-1], device=dev) for v in (f, fp, fpp))
    out = np.zeros(len(ks))
    for i, k in enumerate(ks):
        m = max(1, int(k * float((b - a).max()) / 2.0) + 1)
        edge = torch.arange(m, device=dev, dtype=torch.float64) / m
        u = (edge[:, None] + (xg + 1) / (2 * m)).reshape(-1)      # nodes of [0, 1]
        w = (wg / (2 * m)).repeat(m)
        h = (b - a)[:, None]
        s = h * u
        q = F[:, None] + Fp[:, None] * s + 0.5 * Fpp[:, None] * s * s
        z = k * (a[:, None] + s)
        iz = 1 / z
        sn, cs = torch.sin(z), torch.cos(z)
        z2 = z * z
        if case["nu"] == 2:
            j = (3 * iz * iz - 1) * sn * iz - 3 * cs * iz * iz
            small = z2 / 15 * (1 - z2 / 14 * (1 - z2 / 36 * (1 - z2 / 66 * (1 - z2 / 104 * (1 - z2 / 150)))))
        else:
            j = (15 * iz ** 3 - 6 * iz) * sn * iz - (15 * iz * iz - 1) * cs * iz
            small = z2 * z / 105 * (1 - z2 / 18 * (1 - z2 / 44 * (1 - z2 / 78 * (1 - z2 / 120 * (1 - z2 / 170)))))
        out[i] = float((torch.where(z < 0.7, small, j) * q * w * h).sum())
    return out


def exact(case, seed):
    """C_ℓ sums and Filon integrals in 64 bits.  None for what integrates the hierarchy or recombination: a plain
    64-bit integration of these stiff systems to more digits than the adaptive solver keeps takes minutes."""
    if case["kind"] == "cl":
        return _exact_cl(case, seed)
    if case["kind"] == "filon":
        return _exact_filon(case, seed)
    return None
