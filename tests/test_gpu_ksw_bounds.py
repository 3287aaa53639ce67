"""KSW where the packed kernels' bounds decide, bit-exact against the oracle: N
bonuses and mismatch rewards above the match score, on each side of the 4095
the packed strips hold and of the 65535 the packed row holds."""
import numpy as np
import pytest

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
