"""GPU parity of BANDED in packed halves (two strips a sweep), bit-exact against
the oracle and the 32-bit lanes: odd and even strip counts, word ranges that begin,
end or are empty in one strip of a sweep only, bands from no word to the whole
matrix, scores on each side of the 16-bit bound."""
import numpy as np
import pytest

import gasal2_amd as g
from parity import assert_parity, assert_same, fields, run_both

pytestmark = pytest.mark.gpu


def check(b, **kw):
    runs = []
    for mode in (1, 0):
        g.lib().gasal2_set_pk16(mode)
        try:
            got, ref = run_both(b, g.BANDED, g.WITHOUT_START, False, **kw)
        finally:
            g.lib().gasal2_set_pk16(1)
        assert_parity(got, ref, g.BANDED, g.WITHOUT_START, False, b)
        runs.append(got)
    assert_same(runs[0], runs[1], fields(g.BANDED, g.WITHOUT_START, False), "32-bit lanes")


def mixed(seed, n, longest):
    rng = np.random.default_rng(seed)
    qs, ts = [], []
    for k in range(n):
        t = rng.choice(list(b"ACGT"), int(rng.integers(1, longest))).astype(np.uint8)
        q = t[:max(1, len(t) - int(rng.integers(0, 40)))].copy()
        q[rng.random(len(q)) < 0.06] = ord("T" if k % 3 else "N")
        if len(q) > 24 and k % 2:
            q = np.delete(q, range(12, 15))
        if k % 5 == 0:
            q, t = t, q
        qs.append(q.tobytes())
        ts.append(t.tobytes())
    return g.make_batch(qs, ts)


@pytest.mark.parametrize("k_band", [0, 8, 16, 24, 64, 400])
def test_mixed_shapes(k_band):
    check(mixed(5100 + k_band, 333, 300), k_band=k_band, n_penalty=1)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 200])
def test_batch_sizes(n):
    check(g.synth_batch(4, 5200 + n, n), k_band=32)


@pytest.mark.parametrize("scores", [(1, 4, 6, 1), (2, 3, 5, 2), (7, 8, 0, 1)])
def test_scores(scores):
    check(g.synth_batch(4, 5300, 300), k_band=40, scores=scores, n_penalty=1)


@pytest.mark.parametrize("length", [1160, 1180])
def test_score_bound(length):
    """Identical pairs that score just below and just above 8191 (match 7)."""
    q = bytes(np.random.default_rng(5400).choice(list(b"ACGT"), length).tolist())
    check(g.make_batch([q, q[:100]], [q, q[:90]]), k_band=64, scores=(7, 2, 3, 1))
