"""KSW where the packed kernels' bounds decide, bit-exact against the oracle: N
bonuses and mismatch rewards above the match score, on each side of the 4095
the packed strips hold and of the 65535 the packed row holds; empty queries and
targets, whole waves of them included; one long target among short ones."""
import numpy as np
import pytest
import torch

import gasal2_amd as g
import pyoracle as O

pytestmark = pytest.mark.gpu

FIELDS = ("score", "qend", "tend")


def check(b, scores, n_penalty):
    a = g.Aligner(g.Parameters(algo=g.KSW), int(b.qlen.max()), int(b.tlen.max()), b.n, scores=scores, n_penalty=n_penalty)
    try:
        got = a.run(b)
    finally:
        a.close()
    ref = O.align(b, g.KSW, scores=scores, n_penalty=n_penalty)
    for f in FIELDS:
        assert np.array_equal(got[f], ref[f]), (f, got[f], ref[f])
    return got


@pytest.mark.parametrize("length", [570, 580, 581, 600, 9300, 9400])
@pytest.mark.parametrize("kind", ["n_bonus", "mismatch_reward"])
def test_scores_above_the_match(kind, length):
    """A gap extension as large as the reward keeps every pair off the list of
    pairs the packed strips hand back."""
    q, t = (b"N" * length,) * 2 if kind == "n_bonus" else (b"A" * length, b"T" * length)
    scores, n_penalty = ((1, 4, 7, 7), -7) if kind == "n_bonus" else ((1, -7, 7, 7), None)
    b = g.make_batch([q, b"ACGTACGTAC"], [t, b"ACGTACGTTACC"], seeds=np.array([30, 12], np.uint32))
    assert check(b, scores, n_penalty)["score"][0] == 30 + 7 * length


@pytest.mark.parametrize("empty", [1, 63, 64, 65, 200])
def test_empty_sequences(empty):
    """Sorted last, 64 and more empty queries have a wave to themselves."""
    rng = np.random.default_rng(9100 + empty)
    qs = [rng.choice(list(b"ACGT"), int(rng.integers(1, 90))).astype(np.uint8).tobytes() for _ in range(64)]
    ts = [q[: len(q) // 2] + b"A" + q[len(q) // 2:] for q in qs]
    qs += [b""] * empty + [b"ACGT", b"ACGTACGTA"]
    ts += [b"ACGTACGTAC" * int(rng.integers(1, 9)) if k % 3 else b"" for k in range(empty)] + [b"", b"ACGTACGTA"]
    check(g.make_batch(qs, ts, seeds=rng.integers(0, 40, len(qs)).astype(np.uint32)), (1, 4, 6, 1), 1)


def test_memory_of_one_long_target():
    """40,000 short pairs and a target of 100,000 bases: nothing is sized by the
    number of pairs times the longest target (2 GB of words)."""
    rng = np.random.default_rng(9300)
    t = rng.choice(list(b"ACGT"), 100_000).astype(np.uint8)
    qs = [t[o:o + 40].tobytes() for o in rng.integers(0, 1000, 40_000)]
    ts = [q[:25] + b"AC" + q[25:] for q in qs]
    ts[777] = t.tobytes()
    b = g.make_batch(qs, ts, seeds=rng.integers(0, 30, 40_000).astype(np.uint32))
    a = g.Aligner(g.Parameters(algo=g.KSW), 40, 100_000, b.n)
    try:
        a.load(b, per_pair=False)
        free = torch.cuda.mem_get_info()[0]
        a.run_resident()
        a.sync()
        took = free - torch.cuda.mem_get_info()[0]
        got = a.download()
    finally:
        a.close()
    assert took < 3e8, took
    ref = O.align(b, g.KSW)
    for f in FIELDS:
        assert np.array_equal(got[f], ref[f]), f


@pytest.mark.parametrize("scores", [(1, 4, 6, 1), (1, 4, 2, 8), (2, 3, 0, 3), (3, 2, 5, 0)])
@pytest.mark.parametrize("top_seed", [1, 40, 900])
def test_first_rows_of_long_queries(scores, top_seed):
    """Queries longer than the columns a path can reach in the first sixteen rows,
    related from the start, later or not at all."""
    rng = np.random.default_rng(9400 + top_seed)
    qs, ts = [], []
    for k in range(150):
        q = rng.choice(list(b"ACGT"), int(rng.integers(200, 700))).astype(np.uint8)
        t = rng.choice(list(b"ACGT"), int(rng.integers(20, 300))).astype(np.uint8)
        o = int(rng.integers(0, 60)) if k % 3 else 0
        m = max(min(len(q) - o, len(t)), 0)
        if k % 4:
            t[:m] = q[o:o + m]
            t[rng.random(len(t)) < 0.04] = ord("N")
        qs.append(q.tobytes())
        ts.append(t.tobytes())
    check(g.make_batch(qs, ts, seeds=rng.integers(0, top_seed, 150).astype(np.uint32)), scores, 1)
