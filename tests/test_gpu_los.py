"""The line-of-sight sum at the edges of its splits: x nodes per slot of 64 lanes and
slots per wavefront, chunks of 16 multipoles, the change to the short recurrence at
ℓ = 64, and the spans between two exchanges of a block (256 multipoles with 4 slots a
wavefront, 128 with 1 or 2)."""
import numpy as np
import pytest

import boltmi
import cosmo
import pyoracle
from boltmi import _abi

pytestmark = pytest.mark.gpu


def setting(nxi):
    """tables whose x grid has nxi integration nodes after x = -8, with sources: a bump
    at last scattering, one at reionization and a late smooth part"""
    n = next(n for n in range(16, 4000)
             if sum(cosmo.xnode(j, nx=n) > -8.0 for j in range(n)) - 1 == nxi)
    par = boltmi.CosmoParams()
    bg = boltmi.Background(par, x_grid=(-20.0, 0.0, n))
    k = boltmi.quadratic_k(0.1 * bg.H0, 1000 * bg.H0, 30)
    x = np.asarray(bg.x_grid)
    S = np.exp(-((x + 7.0) / 0.15)**2) + 0.1 * np.exp(-((x + 2.2) / 0.3)**2) + 0.02 * np.exp(x)
    S = S * (1.0 + np.cos(60.0 * k / k[-1]))[:, None]
    P = S / (1.0 + x**2)
    return par, bg, boltmi.SourceGrid(bg.x_grid, k, S), boltmi.SourceGrid(bg.x_grid, k, P), \
        boltmi.quadratic_k(0.01 * bg.H0, 1000 * bg.H0, 520)


# A term is left out where |j_ℓ| is below 1e-7 of its largest value: up to 2e-7 of C_ℓ
# where the sum is of the size of its terms, rounded up to the 1e-6 that the other
# comparisons with the oracle take; 1e-9 of the largest C_ℓ where the terms cancel.
@pytest.mark.parametrize("spw", ["1", "2", "4"])
@pytest.mark.parametrize("nxi", [9, 63, 64, 65, 256, 257, 1024])
def test_x_slots_against_oracle(nxi, spw, monkeypatch):
    monkeypatch.setenv("BOLT_LOS_SPW", spw)
    par, bg, T, P, dense = setting(nxi)
    ctx = boltmi.Context(0)
    ells = np.array([2, 3, 15, 16, 17, 63, 64, 65, 191, 192, 193, 319, 320, 900, 1500])
    o = pyoracle.Oracle(par.as_tuple(), bg.tables_dict())
    got = boltmi.cl_on_grid(ells, T, P, dense, par, bg, ctx=ctx)
    for g, r in zip(got, o.cl(T.grid, P.grid, T.k_grid, dense, ells, 0, nthreads=8)):
        np.testing.assert_allclose(g, r, rtol=1e-6, atol=1e-9 * np.max(np.abs(r)))
    one = boltmi.cltt_on_grid(ells, T, dense, par, bg, ctx=ctx)
    np.testing.assert_allclose(one, got[0], rtol=1e-13)


def test_last_multipole_does_not_matter():
    """C_ℓ is the same to the last bit whatever the largest ℓ of the call is"""
    par, bg, T, P, dense = setting(320)
    full = boltmi.cl_on_grid(np.arange(2, 701), T, P, dense, par, bg)
    tt = boltmi.cltt_on_grid(np.arange(2, 701), T, dense, par, bg)
    for lmax in (2, 15, 16, 17, 63, 64, 65, 79, 80, 191, 192, 193, 320, 321):
        part = boltmi.cl_on_grid(np.arange(2, lmax + 1), T, P, dense, par, bg)
        for g, r in zip(part, full):
            np.testing.assert_array_equal(g, r[:lmax - 1])
        np.testing.assert_array_equal(boltmi.cltt_on_grid(np.arange(2, lmax + 1), T, dense, par, bg), tt[:lmax - 1])


@pytest.mark.parametrize("spw", ["1", "2", "4"])
def test_last_multipole_at_the_end_of_a_span(spw, monkeypatch):
    """the same with the last ℓ at the ends of the spans of 128 and 256, and the values
    there against the oracle (tolerances as above)"""
    monkeypatch.setenv("BOLT_LOS_SPW", spw)
    par, bg, T, P, dense = setting(320)
    ctx = boltmi.Context(0)
    full = boltmi.cl_on_grid(np.arange(2, 531), T, P, dense, par, bg, ctx=ctx)
    tt = boltmi.cltt_on_grid(np.arange(2, 531), T, dense, par, bg, ctx=ctx)
    last = [126, 127, 128, 129, 254, 255, 256, 257, 511, 512, 513]
    for lmax in last:
        part = boltmi.cl_on_grid(np.arange(2, lmax + 1), T, P, dense, par, bg, ctx=ctx)
        for g, r in zip(part, full):
            np.testing.assert_array_equal(g, r[:lmax - 1])
        np.testing.assert_array_equal(boltmi.cltt_on_grid(np.arange(2, lmax + 1), T, dense, par, bg, ctx=ctx),
                                      tt[:lmax - 1])
    o = pyoracle.Oracle(par.as_tuple(), bg.tables_dict())
    ells = np.array([2] + last)
    for g, r in zip(full, o.cl(T.grid, P.grid, T.k_grid, dense, ells, 0, nthreads=8)):
        np.testing.assert_allclose(g[ells - 2], r, rtol=1e-6, atol=1e-9 * np.max(np.abs(r)))
    np.testing.assert_allclose(tt, full[0], rtol=1e-13)


# Both sides sum the same spline terms in 64 bits: 1e-9, as the other comparison with
# the oracle's spline mode.
@pytest.mark.parametrize("nxi,nkd,ells", [
    (9, 2, [2, 3]),                        # one midpoint, fewer columns than a group
    (63, 17, list(range(2, 18))),          # one full tile, one full column group
    (65, 18, list(range(2, 19))),          # a midpoint and a column more
    (320, 65, list(range(0, 34)) + [700]),  # ℓ = 0 and 1, repeated and far ℓ
    (1024, 520, [2, 15, 16, 900, 1500, 15]),
    (320, 161, list(range(2, 513))),       # one column short of a block's last 64
    (320, 161, list(range(2, 514))),       # exactly full
    (256, 161, list(range(2, 700))),       # a partial last block
    (320, 6200, [2, 37, 1100]),            # more midpoints than are kept at once
])
def test_spline_sum_against_oracle(nxi, nkd, ells):
    par, bg, T, P, _ = setting(nxi)
    dense = boltmi.quadratic_k(0.01 * bg.H0, 1000 * bg.H0, nkd)
    ells = np.array(ells)
    o = pyoracle.Oracle(par.as_tuple(), bg.tables_dict())
    got = boltmi.cl_on_grid(ells, T, P, dense, par, bg, bessel_mode=1)
    for g, r in zip(got, o.cl(T.grid, P.grid, T.k_grid, dense, ells, 1, nthreads=8)):
        has = (ells > 0) | np.isfinite(r)  # the oracle's spline mode has no value for ℓ = 0
        assert np.isfinite(g).all()
        np.testing.assert_allclose(g[has], r[has], rtol=1e-9, atol=1e-9 * np.max(np.abs(r[has])))
    np.testing.assert_allclose(boltmi.cltt_on_grid(ells, T, dense, par, bg, bessel_mode=1), got[0], rtol=1e-12)


def test_spline_sum_where_eta_does_not_grow():
    """tables whose η(x) goes back and forth: the x nodes that reach a coefficient are
    no longer contiguous"""
    par, bg, T, P, dense = setting(320)
    x = np.linspace(-20.0, 0.0, bg.nx + 2)
    bg.coef[_abi.T_ETA] *= 1.0 - 0.05 * np.sin(30.0 * x)**2
    ells = np.arange(2, 100)
    o = pyoracle.Oracle(par.as_tuple(), bg.tables_dict())
    eta = np.array([o.spline(_abi.T_ETA, v) for v in bg.x_grid])
    assert (np.diff(eta[bg.x_grid > -8.0]) < 0).any()
    got = boltmi.cl_on_grid(ells, T, P, dense, par, bg, bessel_mode=1)
    for g, r in zip(got, o.cl(T.grid, P.grid, T.k_grid, dense, ells, 1, nthreads=8)):
        np.testing.assert_allclose(g, r, rtol=1e-9, atol=1e-9 * np.max(np.abs(r)))


# |z| = k (η − η₀) <= 0.02 at the one node beyond η₀, where the oracle's j₀ and j₁ are exact
# to rounding; all other nodes at this x have z > 30 from k = 0.004 on
@pytest.mark.parametrize("spw", ["1", "2", "4"])
@pytest.mark.parametrize("node", [1201, 1250, 1500])
def test_exact_sum_where_eta_passes_eta0(node, spw, monkeypatch):
    """tables in which η(x) exceeds η₀ at a node among others with large z: its
    argument is negative, and j_ℓ(−z) = (−1)^ℓ j_ℓ(z)"""
    monkeypatch.setenv("BOLT_LOS_SPW", spw)
    par, bg, T, P, dense = setting(799)
    eta = bg.coef[_abi.T_ETA]  # node j has coefficients j, j + 1, j + 2 with weights 1/6, 2/3, 1/6
    eta[node + 1] += 1.5 * (bg.eta0 + 0.05 - (eta[node] + 4.0 * eta[node + 1] + eta[node + 2]) / 6.0)
    ells = np.array([2, 3, 10, 30, 47, 48, 63, 64, 100, 300, 700])
    o = pyoracle.Oracle(par.as_tuple(), bg.tables_dict())
    assert [i for i, x in enumerate(bg.x_grid) if o.spline(_abi.T_ETA, x) > bg.eta0] == [node]
    ctx = boltmi.Context(0)
    got = boltmi.cl_on_grid(ells, T, P, dense, par, bg, ctx=ctx)
    for g, r in zip(got, o.cl(T.grid, P.grid, T.k_grid, dense, ells, 0, nthreads=8)):
        np.testing.assert_allclose(g, r, rtol=1e-6, atol=1e-9 * np.max(np.abs(r)))
