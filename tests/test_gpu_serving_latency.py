"""A request in the work queue is solved about as fast as the same modes alone: the
idle workgroups of the persistent launch, which poll for work, do not hold up those
that have some, and it runs in the layout of ordinary states unless a request needs more."""
import time

import numpy as np
import pytest

import boltmi
import cosmo

pytestmark = pytest.mark.gpu


# Few modes, so that most workgroups are idle.  Both sides' medians of 7; with 14 µs
# between an idle workgroup's polls the queue took 1.9 times as long.
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


def test_queue_launch_has_the_layout_of_ordinary_states():
    """P(k) at plin's defaults (n = 473) takes the same time either way; in a launch
    whose layout holds any state it took 1.15 times as long.  Minima of 8."""
    par, bg, ih = cosmo.background("c1")
    ks = np.logspace(-3, np.log10(0.25), 10)
    alone, queue = [], []
    srv = boltmi.Server(hbm_gib=1.0, queue=True)
    try:
        for _ in range(8):
            queue.append(srv.wait(srv.submit_pk(par, k=ks))[1]["solve_ms"])
    finally:
        srv.close()
    for _ in range(8):
        t = time.perf_counter()
        boltmi.plin(ks, par, bg, ih)
        alone.append((time.perf_counter() - t) * 1e3)
    assert min(queue) < 1.08 * min(alone), (queue, alone)


def test_requests_of_every_layout_in_one_queue():
    """Requests whose states the running launch does not hold (more than 16 momentum
    bins, more than 512 rows) among others: all are served, bitwise what they give alone
    with the queue's six scan rows a lane, and again after the queue was idle."""
    ks = np.logspace(-3, np.log10(0.2), 12)
    big = np.logspace(-4, np.log10(0.4), 400)
    plan = [(50, 50, 10, 15), (8, 8, 10, 20), (50, 50, 20, 15), (167, 161, 10, 2), (8, 8, 10, 15), (40, 40, 6, 48)]
    srv = boltmi.Server(hbm_gib=2.0, queue=True)
    try:
        par = cosmo.massive_nq(15)[0]
        big_id = srv.submit_cltt(par, k=big, ell_max=200, nkd=400, ℓᵧ=50, ℓ_ν=50, ℓ_mν=10, reltol=1e-9)
        time.sleep(0.1)  # the launch is running
        rounds = []
        for wait in (0.0, 0.3):
            time.sleep(wait)
            ids = [srv.submit_pk(par, k=ks, ℓᵧ=a, ℓ_ν=b, ℓ_mν=c, n_q=q) for a, b, c, q in plan]
            rounds.append([srv.wait(i)[0] for i in ids])
        got_big = srv.wait(big_id)[0]
        assert srv.queue_info()["served"] == 2 * len(plan) + 1
    finally:
        srv.close()
    mp = pytest.MonkeyPatch()
    mp.setenv("BOLT_SOLVER_SR", "6")
    ctx = boltmi.Context(0)
    mp.undo()
    try:
        for i, (a, b, c, q) in enumerate(plan):
            _, bg, ih, _ = cosmo.massive_nq(q)
            ref = boltmi.plin(ks, par, bg, ih, n_q=q, ℓᵧ=a, ℓ_ν=b, ℓ_mν=c, ctx=ctx)
            for got in rounds:
                np.testing.assert_array_equal(got[i], ref, err_msg=str((a, b, c, q)))
        _, bg, ih, _ = cosmo.massive_nq(15)
        sf = boltmi.source_grid(par, bg, ih, big, None, 50, 1e-9, ℓ_ν=50, ℓ_mν=10, ctx=ctx)
        ref = boltmi.cltt_on_grid(np.arange(2, 201), sf, boltmi.quadratic_k(0.01 * bg.H0, 1000 * bg.H0, 400), par, bg,
                                  ctx=ctx)
        np.testing.assert_array_equal(got_big, ref)
    finally:
        ctx.close()
