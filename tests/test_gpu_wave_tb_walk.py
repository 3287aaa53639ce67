"""The two walks of the packed one-wave traceback path, a lane per pair and a
wave per pair, bit-exact against the oracle and the lane kernels: short paths and
large batches on lanes, long paths of few pairs on waves, paths of gaps."""
import numpy as np
import pytest

import gasal2_amd as g
import pyoracle as O
from parity import assert_parity, assert_same, fields

pytestmark = pytest.mark.gpu

MODES = [(g.LOCAL, False), (g.LOCAL, True), (g.GLOBAL, False)]


def related(seed, n, lq, lt):
    """n pairs of lq[0]..lq[1] and lt[0]..lt[1] bases that share their shorter side, with substitutions and an indel."""
    rng = np.random.default_rng(seed)
    base = rng.choice(list(b"ACGT"), 1 << 16).astype(np.uint8)
    qs, ts = [], []
    for a, b, o, cut in zip(rng.integers(lq[0], lq[1] + 1, n), rng.integers(lt[0], lt[1] + 1, n),
                            rng.integers(0, 1 << 15, n), rng.integers(0, 1 << 15, n)):
        q, t = base[o:o + a].copy(), base[o:o + b]
        q[cut % a] = ord("G")
        k = cut % max(min(a, b) - 3, 1)
        t = np.concatenate([t[:k], t[k + cut % 3:], t[:cut % 3]])
        qs.append(q.tobytes())
        ts.append(t.tobytes())
    return g.make_batch(qs, ts)


def run(b, algo, second, policy, sample):
    g.lib().gasal2_set_dispatch(policy)
    a = g.Aligner(g.Parameters(algo=algo, start_pos=g.WITH_TB, secondBest=g.TRUE if second else g.FALSE),
                  int(b.qlen.max()), int(b.tlen.max()), b.n, n_penalty=1)
    try:
        out = a.run(b, per_pair=False)
        out["cigars"] = [a.cigar(k) for k in sample]
        return out, a.last_paths()
    finally:
        g.lib().gasal2_set_dispatch(0)
        a.close()


@pytest.mark.parametrize("n,lq,lt", [(1, (1, 1), (1, 1)), (700, (1, 24), (1, 24)), (900, (8, 8), (16, 16)),
                                     (40_001, (60, 200), (60, 200)), (300, (20, 40), (900, 1500)),
                                     (300, (900, 1500), (20, 40)), (6, (3000, 4000), (3000, 4000))])
@pytest.mark.parametrize("algo,second", MODES)
def test_walks(algo, second, n, lq, lt):
    b = related(7100 + n, n, lq, lt)
    sample = range(0, n, max(n // 1500, 1))
    (wave, paths), (lane, _) = run(b, algo, second, 3, sample), run(b, algo, second, 2, sample)
    assert paths & 6 == 6
    assert_same(wave, lane, fields(algo, g.WITH_TB, second) + ["n_ops", "cigars"], "lane path")
    few = b.subset(np.arange(0, n, max(n // 1500, 1)))
    ref = O.align(few, algo, start_pos=g.WITH_TB, second_best=second, n_penalty=1)
    got = {f: v[::max(n // 1500, 1)] for f, v in wave.items() if isinstance(v, np.ndarray) and len(v) == n}
    got["cigars"] = wave["cigars"]
    assert_parity(got, ref, algo, g.WITH_TB, second)
