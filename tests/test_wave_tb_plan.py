"""The packed one-wave traceback path's plan holds what its waves claim: the host's
plan for a batch's lengths against a model of the device's order and claims.  Every
store of that path lies inside the claimed iterations, so the plan is what keeps
them inside the buffer."""
import numpy as np
import pytest

import gasal2_amd as g


def shape8(x):
    """The order's bucket of a number of words: 128 exact ones, then 16 an octave."""
    e = np.floor(np.log2(np.maximum(x, 1))).astype(np.int64)
    v = 128 + (e - 7) * 16 + ((x >> np.maximum(e - 4, 0)) & 15)
    return np.where(x < 128, x, np.minimum(v, 255))


def claims(qlens, tlens, lanes, rng):
    """Iterations the waves claim, the pairs of a bucket in any order."""
    q, t = (np.asarray(qlens, np.int64) + 7) // 8, (np.asarray(tlens, np.int64) + 7) // 8
    order = np.lexsort((rng.random(len(q)), -shape8(t), -shape8(q)))
    q, t = q[order], t[order]
    total, at = 0, 0
    for group, pairs in zip((256, 64, 32, 16, 4), lanes):
        a, b = q[at:at + pairs], t[at:at + pairs]
        at += pairs
        if group == 256:
            total += int((((b + 127) // 128) * np.maximum(a, 260) + 256).sum())
            continue
        its = ((b + 2 * group - 1) // (2 * group)) * np.maximum(a, group + 1) + group
        for k in range(0, pairs, 64 // group):
            total += int(its[k:k + 64 // group].max())
    assert at == len(q)
    return total


def lengths(kind, n, rng):
    if kind == "equal":
        return np.full(n, 150), np.full(n, 250)
    if kind == "short":
        return rng.integers(1, 60, n), rng.integers(1, 90, n)
    if kind == "mixed":
        q = np.clip(np.exp(rng.normal(5.8, 0.9, n)), 1, 6000).astype(np.int64)
        return q, np.maximum(q + rng.integers(-50, 51, n), 1)
    if kind == "bucket_edges":   # above 128 words several lengths share a bucket
        return rng.integers(1000, 1200, n), rng.integers(1016, 2400, n)
    if kind == "narrow":
        return rng.integers(1, 30, n), rng.integers(500, 30_000, n)
    q, t = rng.integers(100, 300, n), rng.integers(100, 400, n)   # and one long one
    q[n // 2], t[n // 3] = 9000, 20_000
    return q, t


@pytest.mark.parametrize("n", [1, 3, 17, 130, 1001, 9001])
@pytest.mark.parametrize("kind", ["equal", "short", "mixed", "bucket_edges", "narrow", "outlier"])
def test_plan_holds_the_claims(kind, n):
    rng = np.random.default_rng(6100 + n)
    q, t = lengths(kind, n, rng)
    for n_cu in (1, 16, 256):
        plan, *lanes = g.wave_tb_plan(q, t, n_cu)
        assert sum(lanes) == n
        got = max(claims(q, t, lanes, rng) for _ in range(3))
        assert got <= plan, (kind, n, n_cu, lanes)
        assert plan <= 2 * got + 1000, (kind, n, n_cu, lanes)


def test_lane_counts_occur():
    """The lengths above reach every group width."""
    rng = np.random.default_rng(6200)
    used = np.zeros(5, np.int64)
    for kind in ("equal", "mixed", "narrow", "outlier"):
        for n in (17, 130, 1001, 9001):
            used += np.minimum(g.wave_tb_plan(*lengths(kind, n, rng))[1:], 1)
    assert (used > 0).all(), used
