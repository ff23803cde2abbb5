"""A request in the work queue is solved about as fast as the same modes alone: the
idle workgroups of the persistent launch, which poll for work, do not hold up those
that have some."""
import time

import numpy as np
import pytest

import boltmi
import cosmo

pytestmark = pytest.mark.gpu


# Few modes, so that most workgroups are idle.  Both sides' medians of 7; with 14 µs
# between an idle workgroup's polls the queue took 1.9 times as long.  The
# queue's launch holds any state length, which costs up to 1.2 on its own.
@pytest.mark.parametrize("sizes", [(50, 50, 20, 15), (40, 40, 6, 48)])
def test_queue_solves_as_fast_as_a_launch_of_its_own(sizes):
    par, bg, ih, _ = cosmo.massive_nq(sizes[3])
    ks = np.logspace(-3, np.log10(0.25), 10)
    cfg = dict(ℓᵧ=sizes[0], ℓ_ν=sizes[1], ℓ_mν=sizes[2], n_q=sizes[3])
    alone = []
    for _ in range(8):
        t = time.perf_counter()
        ref = boltmi.plin(ks, par, bg, ih, **cfg)
        alone.append((time.perf_counter() - t) * 1e3)
    queue = []
    srv = boltmi.Server(hbm_gib=1.0, queue=True)
    try:
        for _ in range(8):
            pk, info = srv.wait(srv.submit_pk(par, k=ks, **cfg))
            queue.append(info["solve_ms"])
    finally:
        srv.close()
    np.testing.assert_allclose(pk, ref, rtol=1e-6)
    print(f"alone {np.median(alone[1:]):.1f} ms, queue {np.median(queue[1:]):.1f} ms")
    assert np.median(queue[1:]) < 1.4 * np.median(alone[1:]), (queue, alone)
