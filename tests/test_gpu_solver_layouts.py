"""The FP64 solver at the edges of its layouts: 256, 368 and 512 rows (one or two
owned rows per thread, the vectors' strides), 384 rows (one or two scan passes)
and 16 momentum bins, each side of the line, and the longest state.  States at
five x against the oracle at the parity tests' 1e-6, with its step counts; a
source column (wavefront-per-node dense output) at the same bar."""
import numpy as np
import pytest

import boltmi
import cosmo

pytestmark = pytest.mark.gpu

# (ℓᵧ, ℓ_ν, ℓ_mν, nq) with n = 2ℓᵧ + ℓ_ν + (ℓ_mν + 1) nq + 8
SIZES = {38: (8, 8, 2, 2), 256: (30, 23, 10, 15), 257: (30, 24, 10, 15), 360: (60, 67, 10, 15), 361: (60, 68, 10, 15),
         384: (70, 71, 10, 15), 385: (70, 72, 10, 15), 511: (60, 53, 21, 15), 512: (160, 162, 10, 2),
         513: (160, 163, 10, 2), 525: (167, 161, 10, 2)}


def _check(n, sizes):
    par, bg, ih, o = cosmo.massive_nq(sizes[3])
    cfg = boltmi.hier_cfg(*sizes, 1e-6, 1e-6)
    assert boltmi.state_length(cfg) == n
    xs = np.array([-12.0, -8.0, -7.0, -3.0, 0.0])
    ks = [0.004, 0.04]
    U, _, st = boltmi.boltsolve_batch(par, bg, cfg, ks, xs)
    acc = 0
    for i, k in enumerate(ks):
        ref, ost = o.boltsolve(cosmo.ocfg(*sizes), k, xs)
        acc += ost.accepted
        for j in range(len(xs)):
            err = np.max(np.abs(U[i, j] - ref[j])) / np.max(np.abs(ref[j]))
            assert err < 1e-6, (n, k, xs[j], err)
    assert st["accepted"] == acc
    ref, _ = o.source_column(cosmo.ocfg(*sizes), ks[1])
    S = boltmi.source_grid(par, bg, ih, [ks[1]], None, sizes[0], 1e-6, sizes[1], sizes[2], sizes[3]).grid[0]
    assert np.max(np.abs(S - ref)) < 1e-6 * np.max(np.abs(ref)), n


@pytest.mark.parametrize("n", sorted(SIZES))
def test_layout_edges_match_oracle(n):
    _check(n, SIZES[n])


@pytest.mark.parametrize("nq", [16, 17])
def test_momentum_bins_at_the_layout_line_match_oracle(nq):
    sizes = (12, 12, 8, nq)
    _check(2 * 12 + 12 + 9 * nq + 8, sizes)


@pytest.mark.parametrize("ell_nu", [75, 76])
def test_second_layouts_last_row_matches_oracle(ell_nu):
    _check(293 + ell_nu, (60, ell_nu, 10, 15))
