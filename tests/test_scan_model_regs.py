"""A CPU model of the FP64 solver's substitution in registers (bolt.jl_amd/csrc/solve.hip:
fac_prep, subst_regs) with the kernel's DPP controls: the forward scan toward higher
lanes (row_shr 1, 2, 4, 8; row_bcast 15 and 31; wave_shr 1) and the backward one toward
lower lanes over the same rows (row_shl 1, 2, 4, 8; mirror_bcast15 and 31; wave_shl 1),
the lane maps' multipliers formed ahead, one or two passes of 64·SR rows, the two
second-band corrections.  It must give the sequential forward and back substitution.

Rows past n are not masked: their factors are zero (d = u1 = l1 = 0), so that rows
of zeros come out as zeros and stay so in memory, which the next solve relies on.  A
value that is not finite breaks that -- 0·NaN is a NaN -- so those rows are cleared
after it."""
import numpy as np
import pytest

W = 64
LANE = np.arange(W)


def dpp(v, old, ctrl, rmask=0xF):
    out = old.copy()
    for i in range(W):
        row, src = i // 16, None
        if not (rmask >> row) & 1:
            continue
        if 0x111 <= ctrl <= 0x11F and i % 16 >= ctrl - 0x110:          # row_shr n
            src = i - (ctrl - 0x110)
        elif 0x101 <= ctrl <= 0x10F and i % 16 + (ctrl - 0x100) < 16:  # row_shl n
            src = i + (ctrl - 0x100)
        elif ctrl == 0x142 and row >= 1:                               # row_bcast 15
            src = (row - 1) * 16 + 15
        elif ctrl == 0x143 and row >= 2:                               # row_bcast 31
            src = 31
        elif ctrl == 0x138 and i >= 1:                                 # wave_shr 1
            src = i - 1
        elif ctrl == 0x130 and i + 1 < W:                              # wave_shl 1
            src = i + 1
        if src is not None:
            out[i] = v[src]
    return out


def mirror15(v, ident):
    return np.where(LANE // 16 == 0, v[16], np.where(LANE // 16 == 2, v[48], ident))


def mirror31(v, ident):
    return np.where(LANE < 32, v[32], ident)


FWD = [lambda v, e, c=c: dpp(v, np.full(W, e), c) for c in (0x111, 0x112, 0x114, 0x118)] + \
      [lambda v, e: dpp(v, np.full(W, e), 0x142, 0xA), lambda v, e: dpp(v, np.full(W, e), 0x143, 0xC)]
BWD = [lambda v, e, c=c: dpp(v, np.full(W, e), c) for c in (0x101, 0x102, 0x104, 0x108)] + [mirror15, mirror31]


def rows(vec, p, SR, n):
    """lane_rows: a lane's group is loaded as a whole if its first row is below n"""
    j0 = W * SR * p + SR * LANE
    r = vec[j0[:, None] + np.arange(SR)]
    return np.where((j0 < n)[:, None], r, 0.0)


def multipliers(a, steps):
    out = []
    for f in steps:
        out.append(a)
        a = a * f(a, 1.0)
    return out, a


def solve(l1, d, u1, l2, u2, vec, n, SR):
    """one substitution of vec (rows past n included, as the workspace holds them)"""
    NP = (n + W * SR - 1) // (W * SR)
    F, v = [], []
    for p in range(NP):
        l, dd, u = -rows(l1, p, SR, n), rows(d, p, SR, n), rows(u1, p, SR, n)
        r = -dd[:, ::-1] * u[:, ::-1]
        la, lf = multipliers(np.multiply.reduce(l, axis=1), FWD)
        ra, rf = multipliers(np.multiply.reduce(r, axis=1), BWD)
        F.append((l, r, dd, u, la, lf, ra, rf))
        v.append(rows(vec, p, SR, n))
    carry = 0.0
    for p, (l, _, _, _, la, lf, _, _) in enumerate(F):
        be = v[p].copy()
        if p == 0:
            be[0, 3] -= (l2 * (l[:, 1] * be[:, 0] + be[:, 1]))[0]
        for i in range(1, SR):
            be[:, i] = l[:, i] * be[:, i - 1] + be[:, i]
        B = be[:, SR - 1].copy()
        for a, f in zip(la, FWD):
            B = a * f(B, 0.0) + B
        if p > 0:
            B = lf * carry + B
        tin = dpp(B, np.full(W, carry), 0x138)
        carry = B[W - 1]
        v[p] = np.cumprod(l, axis=1) * tin[:, None] + be
    carry = 0.0
    for p in range(NP - 1, -1, -1):
        _, r, dd, u, _, _, ra, rf = F[p]
        be = dd[:, ::-1] * v[p][:, ::-1]
        y0, y1 = v[0][0, 0], v[0][0, 1]
        for i in range(1, SR):
            be[:, i] = r[:, i] * be[:, i - 1] + be[:, i]
        B = be[:, SR - 1].copy()
        for a, f in zip(ra, BWD):
            B = a * f(B, 0.0) + B
        if p < NP - 1:
            B = rf * carry + B
        tin = dpp(B, np.full(W, carry), 0x130)
        carry = B[0]
        v[p] = (np.cumprod(r, axis=1) * tin[:, None] + be)[:, ::-1]
        if p == 0:
            x1 = ((y1 - u2 * v[0][0, 3]) - u[0, 1] * v[0][0, 2]) * dd[0, 1]
            x0 = (y0 - u[0, 0] * x1) * dd[0, 0]
            v[0][0, 1], v[0][0, 0] = x1, x0
    out = vec.copy()
    for p in range(NP):
        for lane in LANE:  # store_rows: whole groups
            j0 = W * SR * p + SR * lane
            if j0 < n:
                out[j0:j0 + SR] = v[p][lane]
    return out


def sequential(l1, d, u1, l2, u2, b, n):
    y = np.zeros(n)
    for j in range(n):
        y[j] = b[j] - (l1[j] * y[j - 1] if j else 0.0) - (l2 * y[1] if j == 3 else 0.0)
    x = np.zeros(n)
    for j in range(n - 1, -1, -1):
        x[j] = d[j] * (y[j] - (u1[j] * x[j + 1] if j + 1 < n else 0.0) - (u2 * x[3] if j == 1 else 0.0))
    return x


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("n", [38, 197, 198, 256, 323, 384, 385, 448, 473, 512, 525])
@pytest.mark.parametrize("SR", [6, 7, 8])
def test_substitution_in_registers_model(n, SR):
    rng = np.random.default_rng(1000 * n + SR)
    pad = np.zeros(2 * W * SR + SR - n)
    l1, u1, d = (np.concatenate([rng.uniform(a, b, n), pad]) for a, b in ((-1, 1), (-1, 1), (0.5, 2)))
    l1[0] = u1[n - 1] = 0.0
    b = rng.uniform(-1, 1, n)
    vec = np.concatenate([b, pad])
    with np.errstate(all="ignore"):
        got = solve(l1, d, u1, 0.3, -0.2, vec, n, SR)
        ref = sequential(l1, d, u1, 0.3, -0.2, b, n)
        assert np.max(np.abs(got[:n] - ref)) < 1e-14 * np.max(np.abs(ref))
        assert (got[n:] == 0.0).all()
        # after a right-hand side that was not finite: NaNs past n where n ends inside a
        # lane's group; with those cleared the next solve is the first one again
        bad = vec.copy()
        bad[n // 2] = np.nan
        left = solve(l1, d, u1, 0.3, -0.2, bad, n, SR)
        assert np.isnan(left[n:]).any() == (n % SR != 0)
        left[:n] = b
        if n % SR:
            assert np.isnan(solve(l1, d, u1, 0.3, -0.2, left, n, SR)[:n]).any()
        left[n:] = 0.0
        np.testing.assert_array_equal(solve(l1, d, u1, 0.3, -0.2, left, n, SR), got)
