"""The moment tables' prefilter at the edges of its tiles (32 unknowns a lane, 4032 a
block, 48 of warm-up), and the Filon sum at the edges of its 256 lanes, against the
oracle."""
import numpy as np
import pytest

import boltmi
import pyoracle as po

pytestmark = pytest.mark.gpu


# 2e-14 of the moments' scale, as the other comparison of the tables
@pytest.mark.parametrize("n", [4, 5, 33, 34, 35, 49, 50, 51, 4033, 4034, 4035, 4066, 4081, 4082, 4083, 8066, 8067])
def test_prefilter_tiles(n):
    key = (2, 4, 0.0, 120.0, n)
    got, ref = boltmi.sph_bessel_interpolator(*key).coefficients(), po.MomentTable(*key).coefficients()
    xn = np.concatenate([[0.0], np.linspace(0.0, 120.0, n), [120.0]])
    for m in range(4):
        scale = np.maximum(np.abs(ref[m]), np.maximum(1.0, np.maximum(xn, 1.0)**(m - 1.0)))
        assert np.max(np.abs(got[m] - ref[m]) / scale) < 2e-14, m


# 1e-13 of the largest sum, as the other comparison of the sums
@pytest.mark.parametrize("nt", [2, 64, 65, 256, 257, 258, 513])
def test_filon_sum_lanes(nt):
    key = (2, 3, 0.0, 300.0, 30001)
    t = np.linspace(0.05, 12.0, nt)
    f, fp, fpp = np.cos(0.7 * t) + 0.1 * t, -0.7 * np.sin(0.7 * t) + 0.1, -0.49 * np.cos(0.7 * t)
    ks = np.geomspace(0.01, 30.0, 7)
    got = boltmi.filon_sum(boltmi.sph_bessel_interpolator(*key), t, f, fp, fpp, ks)
    ref = po.MomentTable(*key).filon_sum(t, f, fp, fpp, ks)
    assert np.max(np.abs(got - ref)) < 1e-13 * max(1.0, np.max(np.abs(ref)))


# one to four wavefronts a sum: the same 1e-13
@pytest.mark.parametrize("nt", [3, 66, 129, 130, 193, 194])
def test_filon_sum_of_few_intervals(nt):
    key = (2, 3, 0.0, 300.0, 30001)
    t = np.linspace(0.05, 12.0, nt)
    f, fp, fpp = np.cos(0.7 * t) + 0.1 * t, -0.7 * np.sin(0.7 * t) + 0.1, -0.49 * np.cos(0.7 * t)
    ks = np.geomspace(0.01, 30.0, 300)
    got = boltmi.filon_sum(boltmi.sph_bessel_interpolator(*key), t, f, fp, fpp, ks)
    ref = po.MomentTable(*key).filon_sum(t, f, fp, fpp, ks)
    assert np.max(np.abs(got - ref)) < 1e-13 * max(1.0, np.max(np.abs(ref)))
