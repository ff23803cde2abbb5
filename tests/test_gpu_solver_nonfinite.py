"""A trial step whose stages are not finite is rejected and shortened (h to h/5), and
the mode goes on.  Tables with a hole -- one spline coefficient of τ′ a NaN, 0.04 wide
in x -- make steps that would touch it fail; shorter ones land before it, and a later
one passes over it with no stage point inside, as in the oracle: the same accepted
and rejected steps, and states at the parity tests' 1e-6."""
import numpy as np
import pytest

import boltmi
import cosmo
import pyoracle
from boltmi import _abi

pytestmark = pytest.mark.gpu

K = 5e-4          # outside the horizon until late: steps of 0.05..0.3 in x
HOLE = 251        # coefficient of the node x = -17.5
XS = np.array([-12.0, 0.0])


# sizes of every LDS layout: rows that end inside a lane's group of 6, 7 or 8 and rows
# that do not, one and two scan passes
@pytest.mark.parametrize("sr", ["6", "7", "8"])
@pytest.mark.parametrize("sizes", [(8, 8, 10, 15), (30, 23, 10, 15), (50, 50, 10, 15), (50, 50, 20, 15),
                                   (12, 12, 8, 17), (167, 161, 10, 2)])
def test_a_mode_recovers_from_a_nonfinite_step(sizes, sr, monkeypatch):
    par = cosmo.massive_nq(sizes[3])[0]
    bg = boltmi.Background(par, nq=sizes[3])
    boltmi.IonizationHistory(boltmi.RECFAST(bg), par, bg)
    smooth = pyoracle.Oracle(par.as_tuple(), bg.tables_dict()).boltsolve(cosmo.ocfg(*sizes), K, XS)[1]
    bg.coef[_abi.T_TAU_P][HOLE] = np.nan
    ref, st = pyoracle.Oracle(par.as_tuple(), bg.tables_dict()).boltsolve(cosmo.ocfg(*sizes), K, XS)
    assert st.status == 0 and np.isfinite(ref).all()
    assert (st.accepted, st.rejected) != (smooth.accepted, smooth.rejected)  # the hole was met
    monkeypatch.setenv("BOLT_SOLVER_SR", sr)
    ctx = boltmi.Context(0)
    try:
        U, status, got = boltmi.boltsolve_batch(par, bg, boltmi.hier_cfg(*sizes, 1e-6, 1e-6), [K], XS, ctx=ctx)
    finally:
        ctx.close()
    assert status[0] == 0
    assert (got["accepted"], got["rejected"]) == (st.accepted, st.rejected)
    for j in range(len(XS)):
        assert np.max(np.abs(U[0, j] - ref[j])) < 1e-6 * np.max(np.abs(ref[j]))
