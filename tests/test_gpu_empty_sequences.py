"""Pairs with an empty query or target among others, under every dispatch policy,
bit-exact against the oracle; waves of empty pairs included."""
import numpy as np
import pytest

import gasal2_amd as g
import pyoracle as O
from parity import assert_parity

pytestmark = pytest.mark.gpu


def batch(seed, n, empty):
    """n pairs, `empty` of them with no query, no target or neither, first pairs full."""
    rng = np.random.default_rng(seed)
    qs, ts = [], []
    for k in range(n):
        q = rng.choice(list(b"ACGT"), int(rng.integers(1, 120))).astype(np.uint8).tobytes()
        t = q[:len(q) // 2] + b"GA" + q[len(q) // 2:]
        if k >= n - empty:
            q, t = [(b"", t), (q, b""), (b"", b"")][k % 3]
        qs.append(q)
        ts.append(t)
    return g.make_batch(qs, ts)


def check(algo, start, second, tail, policy, scores=(1, 4, 6, 1)):
    for n, empty in ((3, 1), (70, 5), (300, 200)):
        b = batch(9900 + n, n, empty)
        g.lib().gasal2_set_dispatch(policy)
        try:
            a = g.Aligner(g.Parameters(algo=algo, start_pos=start, secondBest=g.TRUE if second else g.FALSE,
                                       semiglobal_skipping_tail=tail, k_band=24),
                          int(b.qlen.max()), int(b.tlen.max()), b.n, scores=scores, n_penalty=1)
            got = a.run(b)
            if start == g.WITH_TB:
                got["cigars"] = [a.cigar(k) for k in range(b.n)]
            a.close()
        finally:
            g.lib().gasal2_set_dispatch(0)
        ref = O.align(b, algo, start_pos=start, second_best=second, tail=tail, k_band=24, scores=scores, n_penalty=1)
        assert_parity(got, ref, algo, start, second)


@pytest.mark.parametrize("scores", [(1, 4, 6, 1), (0, 1, 1, 1), (7, 8, 0, 1)])
@pytest.mark.parametrize("policy", [0, 1, 2, 3])
@pytest.mark.parametrize("second", [False, True])
def test_local_walk(second, policy, scores):
    """A pair without cells: the walk reads its first cell as 0, one match."""
    check(g.LOCAL, g.WITH_TB, second, g.TARGET, policy, scores)


@pytest.mark.parametrize("policy", [0, 1, 2, 3])
@pytest.mark.parametrize("algo,start,second", [(g.LOCAL, g.WITHOUT_START, False), (g.LOCAL, g.WITH_START, False),
                                               (g.LOCAL, g.WITHOUT_START, True), (g.GLOBAL, g.WITHOUT_START, False),
                                               (g.GLOBAL, g.WITH_TB, False), (g.SEMI_GLOBAL, g.WITHOUT_START, False),
                                               (g.SEMI_GLOBAL, g.WITHOUT_START, True), (g.SEMI_GLOBAL, g.WITH_START, False),
                                               (g.SEMI_GLOBAL, g.WITH_START, True), (g.BANDED, g.WITHOUT_START, False)])
def test_scores(algo, start, second, policy):
    """The packed lane kernels took the end of a query without columns from the strips' boundary."""
    for tail in (g.NONE, g.TARGET, g.BOTH) if algo == g.SEMI_GLOBAL else (g.TARGET,):
        check(algo, start, second, tail, policy)
