"""N bonuses and mismatch rewards above the match score where the packed kernels'
bounds decide, bit-exact against the oracle: the one-lane kernels (policy 2) and
the automatic choice, lengths below and above 4095, above 8191 and above
32767 at 7 a cell."""
import numpy as np
import pytest

import gasal2_amd as g
from parity import assert_parity, run_both

pytestmark = pytest.mark.gpu

MODES = [(g.LOCAL, g.WITHOUT_START, False), (g.LOCAL, g.WITH_START, False), (g.LOCAL, g.WITH_TB, False),
         (g.LOCAL, g.WITHOUT_START, True), (g.LOCAL, g.WITH_TB, True), (g.GLOBAL, g.WITHOUT_START, False),
         (g.GLOBAL, g.WITH_TB, False), (g.SEMI_GLOBAL, g.WITHOUT_START, False), (g.SEMI_GLOBAL, g.WITH_START, False),
         (g.BANDED, g.WITHOUT_START, False)]


@pytest.mark.parametrize("kind", ["n_bonus", "mismatch_reward"])
@pytest.mark.parametrize("algo,start,second", MODES)
def test_scores_above_the_match(algo, start, second, kind):
    rng = np.random.default_rng(9500)
    a, c, n_penalty, scores = ("N", "N", -7, (1, 4, 6, 1)) if kind == "n_bonus" else ("A", "T", None, (1, -7, 6, 1))
    for length in (580, 590, 1175) + ((4700,) if not second and start != g.WITH_TB else ()):
        qs, ts = [], []
        for cut in (0, 40):
            q, t = a * length, c * (length - cut)
            qs.append((q[:length // 2] + "GATTACA" + q[length // 2:length - 7]).encode())
            ts.append(t.encode())
        qs.append(rng.choice(list(b"ACGT"), 90).astype(np.uint8).tobytes())
        ts.append(qs[-1][10:80])
        b = g.make_batch(qs, ts)
        for policy in (0, 2):
            g.lib().gasal2_set_dispatch(policy)
            try:
                got, ref = run_both(b, algo, start, second, k_band=4800, scores=scores, n_penalty=n_penalty)
            finally:
                g.lib().gasal2_set_dispatch(0)
            assert_parity(got, ref, algo, start, second)
