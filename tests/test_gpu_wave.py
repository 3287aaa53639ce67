"""GPU parity of the packed one-wave path (16 or 64 lanes per pair) in the score
and start modes, bit-exact against the oracle and against the lane kernels.
Shapes cross its edges: 256-row (16 lanes) and 1024-row (64 lanes) passes, odd
strip counts, queries shorter than a pass is deep, single bases, four pairs of
unlike size in one wave, and scores on both sides of the ranked-cell bound."""
import numpy as np
import pytest

import gasal2_amd as g
from parity import assert_parity, assert_same, fields, run_both

pytestmark = pytest.mark.gpu

EDGES = [(1, 1), (8, 8), (9, 7), (150, 256), (150, 257), (16, 300), (3, 700), (700, 3), (250, 248), (250, 512),
         (301, 520), (64, 1024), (70, 1025), (1100, 1030), (520, 2050), (255, 9), (40, 263), (33, 249)]


def edge_batch(seed, n_rate=0.01):
    rng = np.random.default_rng(seed)
    qs, ts = [], []
    for lq, lt in EDGES * 2:
        q = rng.choice(list(b"ACGT"), lq).astype(np.uint8)
        t = rng.choice(list(b"ACGT"), lt).astype(np.uint8)
        m = min(lq, lt)
        o = int(rng.integers(0, lt - m + 1))
        t[o:o + m] = q[:m]                       # a shared stretch, then substitutions and an indel
        t[rng.random(lt) < 0.04] = ord("G")
        if lt > 40:
            cut = int(rng.integers(10, lt - 10))
            t = np.concatenate([t[:cut], t[cut + 2:], t[:2]])
        for s in (q, t):
            s[rng.random(len(s)) < n_rate] = ord("N")
        qs.append(q.tobytes())
        ts.append(t.tobytes())
    return g.make_batch(qs, ts)


def both_paths(b, algo, start, **kw):
    """The batch with every pair on the one-wave path, then one lane per pair."""
    L = g.lib()
    runs = []
    for policy in (3, 2):
        L.gasal2_set_dispatch(policy)
        try:
            got, ref = run_both(b, algo, start, False, **kw)
        finally:
            L.gasal2_set_dispatch(0)
        assert_parity(got, ref, algo, start, False, b)
        runs.append(got)
    assert_same(runs[0], runs[1], fields(algo, start, False), "lane path")


MODES = [(g.LOCAL, g.WITHOUT_START), (g.LOCAL, g.WITH_START), (g.GLOBAL, g.WITHOUT_START),
         (g.SEMI_GLOBAL, g.WITHOUT_START), (g.SEMI_GLOBAL, g.WITH_START)]


@pytest.mark.parametrize("scores", [(1, 4, 6, 1), (2, 3, 5, 2), (7, 8, 0, 1)])
@pytest.mark.parametrize("algo,start", MODES)
def test_edges(algo, start, scores):
    both_paths(edge_batch(3100 + scores[0]), algo, start, scores=scores, n_penalty=1)


@pytest.mark.parametrize("head", [g.NONE, g.QUERY, g.TARGET, g.BOTH])
@pytest.mark.parametrize("tail", [g.NONE, g.QUERY, g.TARGET, g.BOTH])
def test_semi_heads_and_tails(head, tail):
    for b, rc in ((edge_batch(3200), False), (g.synth_batch(2, 3201, 257), True)):
        for start in (g.WITHOUT_START, g.WITH_START):
            both_paths(b, g.SEMI_GLOBAL, start, head=head, tail=tail, is_rc=rc)


@pytest.mark.parametrize("algo,start", MODES)
def test_mixed_lengths_default_policy(algo, start):
    """Log-normal lengths under the automatic policy: a batch of long pairs
    takes the one-wave path (bit 1 of gasal2_last_paths)."""
    b = g.synth_batch(3, 3300, 130)
    got, ref = run_both(b, algo, start, False)
    assert_parity(got, ref, algo, start, False, b)
    p = g.Parameters(algo=algo, start_pos=start)
    a = g.Aligner(p, int(b.qlen.max()), int(b.tlen.max()), b.n)
    try:
        a.run(b)
        assert a.last_paths() & 2
    finally:
        a.close()


@pytest.mark.parametrize("length,scores", [(1150, (7, 2, 3, 1)), (1190, (7, 2, 3, 1)), (4500, (7, 2, 3, 1)),
                                           (4700, (7, 2, 3, 1))])
def test_local_score_bounds(length, scores):
    """Identical pairs whose score lies on each side of 8191 (cells ranked with
    their row) and of 32000 (packed halves)."""
    rng = np.random.default_rng(3400 + length)
    q = bytes(rng.choice(list(b"ACGT"), length).tolist())
    b = g.make_batch([q, q[: length // 2], b"ACGT" * 60], [q, q[length // 3:], b"TTACGT" * 50])
    both_paths(b, g.LOCAL, g.WITH_START, scores=scores)
    both_paths(b, g.LOCAL, g.WITHOUT_START, scores=scores)


@pytest.mark.parametrize("algo,start", MODES)
def test_no_score_tables(algo, start):
    """Nibbles that share a score-table class ('I' and 'A'): the lane kernels run."""
    b = edge_batch(3500)
    q = bytearray(b.query(3))
    q[5:7] = b"IA"
    b = g.make_batch([bytes(q)] + [b.query(i) for i in range(1, b.n)], [b.target(i) for i in range(b.n)])
    both_paths(b, algo, start)
