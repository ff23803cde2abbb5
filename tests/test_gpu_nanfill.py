"""No k-mode reads a value of its workspace that it did not write: the debug library,
whose solver fills the workspace with NaNs before every mode, gives what the library
gives, bit for bit.  Every LDS layout of the FP64 solver, sources and states from the
starting point on, the FP32 and tangent solves, and modes from the work queue."""
import os
import subprocess
import sys

if __name__ == "__main__":
    import torch  # noqa: F401  (before the library: both then use torch's HIP runtime)
    _root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    sys.path[:0] = [os.path.join(_root, d) for d in ("bolt.jl_amd", "oracle", "tests")]

import numpy as np
import pytest

import boltmi
import cosmo

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(boltmi.__file__))), "libbolt_hip_nanfill.so")


def modes():
    out = {}
    xs = np.array([-20.0, -19.99, -8.0, 0.0])
    ks = np.array([0.003, 0.05])
    for sizes in ((8, 8, 10, 15), (50, 50, 10, 15), (50, 50, 20, 15), (12, 12, 8, 17), (167, 161, 10, 2)):
        par = cosmo.massive_nq(sizes[3])[0]
        bg = boltmi.Background(par, nq=sizes[3])
        ih = boltmi.IonizationHistory(boltmi.RECFAST(bg), par, bg)
        cfg = boltmi.hier_cfg(*sizes, 1e-6, 1e-6)
        n = boltmi.state_length(cfg)
        out[f"u{n}_{sizes[3]}"] = boltmi.boltsolve_batch(par, bg, cfg, ks, xs)[0]
        T, P = boltmi.source_grid_batch([(par, bg, ih)], ks, ℓᵧ=sizes[0], ℓ_ν=sizes[1], ℓ_mν=sizes[2], nq=sizes[3],
                                        reltol=1e-6, want_p=True)
        out[f"s{n}_{sizes[3]}"], out[f"p{n}_{sizes[3]}"] = T[0].grid, P[0].grid
    par, bg, ih = cosmo.background("massive")
    cfg = boltmi.hier_cfg(8, 8, 10, 15, 1e-6, 1e-6)
    cfg.flags |= boltmi.FP32_SOLVE
    out["fp32"] = boltmi.boltsolve_batch(par, bg, cfg, ks, xs)[0]
    dpar = boltmi.CosmoParams(Ω_b=boltmi.Dual(0.046, 1.0))
    dbg = boltmi.Background(dpar)
    dih = boltmi.IonizationHistory(boltmi.RECFAST(dbg), dpar, dbg)
    sf = boltmi.source_grid(dpar, dbg, dih, ks, None, 8, 1e-6).grid
    out["jv"], out["jd"] = sf.v, sf.d
    srv = boltmi.Server(hbm_gib=1.0, queue=True)
    try:
        ids = {l: srv.submit_pk(par, k=ks, ℓᵧ=l, ℓ_ν=l) for l in (8, 30, 50)}
        out.update({f"q{l}": srv.wait(i)[0] for l, i in ids.items()})
    finally:
        srv.close()
    return out


def test_modes_from_a_workspace_of_nans_are_the_same(tmp_path):
    csrc = os.path.join(os.path.dirname(LIB), "csrc")
    if not os.path.exists(LIB) or any(os.path.getmtime(os.path.join(csrc, f)) > os.path.getmtime(LIB)
                                      for f in os.listdir(csrc)):
        pytest.skip("libbolt_hip_nanfill.so is not built from these sources (build.py --nanfill)")
    path = str(tmp_path / "nanfill.npz")
    subprocess.run([sys.executable, os.path.abspath(__file__), path], env=dict(os.environ, BOLT_HIP_LIB=LIB), check=True,
                   timeout=100)
    ref = modes()
    with np.load(path) as got:
        assert sorted(got.files) == sorted(ref)
        for name in ref:
            assert not np.isnan(ref[name]).any(), name  # (the polarization source is infinite at x = 0)
            np.testing.assert_array_equal(got[name], ref[name], err_msg=name)


if __name__ == "__main__":
    np.savez(sys.argv[1], **modes())
