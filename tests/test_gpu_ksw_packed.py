"""GPU parity of KSW in packed strips (the reference's form), bit-exact against
the oracle and against the row by row kernel: query and target lengths on each
side of whole words and of sixteen-row strips, seeds from 0 up, pairs whose rows
die, die early under a live left boundary, or outrun the row above (those the
packed kernel hands back), and settings on each side of its conditions."""
import numpy as np
import pytest

import gasal2_amd as g
import pyoracle as O

pytestmark = pytest.mark.gpu

FIELDS = ("score", "qend", "tend")


def run(b, scores, pk16, n_penalty=1, rc=False):
    L = g.lib()
    L.gasal2_set_pk16(pk16)
    try:
        p = g.Parameters(algo=g.KSW, isReverseComplement=rc)
        a = g.Aligner(p, int(b.qlen.max()), int(b.tlen.max()), b.n, scores=scores, n_penalty=n_penalty)
        try:
            return a.run(b)
        finally:
            a.close()
    finally:
        L.gasal2_set_pk16(1)


def check(b, scores=(1, 4, 6, 1), n_penalty=1, end_bonus=5, rc=False):
    g.set_ksw_extension(end_bonus=end_bonus)
    try:
        packed, rows = run(b, scores, 1, n_penalty, rc), run(b, scores, 0, n_penalty, rc)
    finally:
        g.set_ksw_extension()
    ref = O.align(b, g.KSW, scores=scores, n_penalty=n_penalty, ksw_end_bonus=end_bonus, is_rc=rc)
    for f in FIELDS:
        bad = np.nonzero(packed[f] != ref[f])[0]
        assert len(bad) == 0, (f, len(bad), int(bad[0]), b.query(bad[0]), b.target(bad[0]), int(b.seeds[bad[0]]),
                               int(packed[f][bad[0]]), int(ref[f][bad[0]]))
        assert np.array_equal(rows[f], ref[f]), f


def pairs(seed, n, kind, max_len=120):
    rng = np.random.default_rng(seed)
    qs, ts = [], []
    for _ in range(n):
        lq, lt = int(rng.integers(1, max_len)), int(rng.integers(1, max_len))
        q = rng.choice(list(b"ACGT"), lq).astype(np.uint8)
        t = rng.choice(list(b"ACGT"), lt).astype(np.uint8)
        if kind != "unrelated":
            m = min(lq, lt)
            t[:m] = q[:m]
            if kind == "gaps" and lt > 30:   # long deletions and insertions
                at, cut = int(rng.integers(5, lt - 15)), int(rng.integers(1, 14))
                t = np.concatenate([t[:at], t[at + cut:], t[:cut]]) if rng.random() < 0.5 else \
                    np.concatenate([t[:at], rng.choice(list(b"ACGT"), cut).astype(np.uint8), t[at:lt - cut]])
            if kind == "dies" and lt > 12:   # unrelated from some row on
                at = int(rng.integers(2, lt - 4))
                t[at:] = rng.choice(list(b"ACGT"), lt - at)
            sub = rng.random(lt) < 0.05
            t[sub] = rng.choice(list(b"ACGTN"), int(sub.sum()))
        qs.append(q.tobytes())
        ts.append(t.tobytes())
    seeds = rng.integers(0, 30, n).astype(np.uint32)
    return g.make_batch(qs, ts, seeds=seeds)


@pytest.mark.parametrize("kind", ["related", "gaps", "dies", "unrelated"])
@pytest.mark.parametrize("scores", [(1, 4, 6, 1), (2, 3, 5, 2), (7, 1, 5, 0), (3, 8, 0, 1)])
def test_kinds(kind, scores):
    check(pairs(4200 + scores[0], 1500, kind), scores, end_bonus=min(5, scores[2] + scores[3]))


@pytest.mark.parametrize("end_bonus", [0, 5, 7, 8, 100])
def test_end_bonus(end_bonus):
    check(pairs(4300, 1500, "related"), end_bonus=end_bonus)


@pytest.mark.parametrize("n", [1, 63, 65])
def test_whole_words_and_long_queries(n):
    rng = np.random.default_rng(4400 + n)
    qs, ts = [], []
    for k in range(n):
        lq = int(rng.choice([8, 16, 64, 120, 128, 248, 1023, 1024]))
        q = rng.choice(list(b"ACGT"), lq).astype(np.uint8).tobytes()
        qs.append(q)
        ts.append(q[:5] + b"TT" + q[5:] if k % 2 else q[: lq - 1] + b"GATTACA" * (k % 4))
    check(g.make_batch(qs, ts, seeds=rng.integers(0, 60, n).astype(np.uint32)))


def test_seed_workload_and_score_bound():
    b = g.synth_batch(4, 4500, 3001)
    check(b)
    b.seeds[7] = 3900    # above 4095 with the matches: the row by row kernel
    check(b)


def test_reversed_pairs_and_no_score_tables():
    b = pairs(4600, 700, "related")
    b.qop[::2], b.top[::3] = 3, 1
    check(b, rc=True)
    q = bytearray(b.query(2))
    q[0:2] = b"IA"
    b = g.make_batch([b.query(0), b.query(1), bytes(q)] + [b.query(i) for i in range(3, b.n)],
                     [b.target(i) for i in range(b.n)], seeds=b.seeds)
    check(b)
