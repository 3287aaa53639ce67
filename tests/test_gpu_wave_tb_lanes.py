"""Which lanes WITH_TB on the packed one-wave path ran a batch on, at the edges of
each group's passes and where one group takes many passes, bit-exact against the
oracle and the lane kernels; the iterations its waves claim lie within the plan.
And which of the packed kernels the other modes took or left."""
import numpy as np
import pytest

import gasal2_amd as g
import pyoracle as O
from parity import assert_parity, assert_same, fields
from test_gpu_wave_tb_walk import related

pytestmark = pytest.mark.gpu

MODES = [(g.LOCAL, False), (g.LOCAL, True), (g.GLOBAL, False)]


def run(b, algo, second, policy, sample):
    g.lib().gasal2_set_dispatch(policy)
    a = g.Aligner(g.Parameters(algo=algo, start_pos=g.WITH_TB, secondBest=g.TRUE if second else g.FALSE),
                  int(b.qlen.max()), int(b.tlen.max()), b.n, n_penalty=1)
    try:
        out = a.run(b, per_pair=False)
        out["cigars"] = [a.cigar(k) for k in sample]
        return out, a.last_wave_tb()
    finally:
        g.lib().gasal2_set_dispatch(0)
        a.close()


def edges(strips, words, copies=4):
    """Pairs of `strips` target strips, each less 0 to 7 rows, `words` query words, less 0 to 7 columns."""
    rng = np.random.default_rng(7300 + strips[0])
    qs, ts = [], []
    for s in strips * copies:
        for w in words:
            t = rng.choice(list(b"ACGT"), 8 * s - int(rng.integers(0, 8))).astype(np.uint8)
            q = rng.choice(list(b"ACGT"), 8 * w - int(rng.integers(0, 8))).astype(np.uint8)
            m = min(len(q), len(t))
            o = int(rng.integers(0, len(t) - m + 1))
            q[:m] = t[o:o + m]
            q[rng.random(len(q)) < 0.05] = ord("C")
            cut = len(q) // 2
            qs.append(np.concatenate([q[:cut], q[cut + 3:], q[:3]]).tobytes())
            ts.append(t.tobytes())
    return g.make_batch(qs, ts)


# lanes of the whole batch (index into 256, 64, 32, 16, 4), the batch
CASES = {
    "64 lanes, a pass and one strip less": (1, lambda: edges([127, 128], [64, 65, 70])),
    "32 lanes, a pass and one strip less and more": (2, lambda: edges([63, 64, 65], [30, 31, 33, 40])),
    "32 lanes, queries shorter than the lag of its lanes": (2, lambda: edges([64], [26, 27, 28])),
    "32 lanes, two passes": (2, lambda: edges([127, 128, 129], [34, 36])),
    "16 lanes, a pass and one strip less and more": (3, lambda: edges([31, 32, 33], [18, 19, 22])),
    "4 lanes, one to thirteen passes": (4, lambda: related(7400, 60_001, (130, 160), (1, 800))),
    "4 lanes, seven passes": (4, lambda: related(7401, 30_001, (160, 210), (380, 400))),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("algo,second", MODES)
def test_lanes(algo, second, name):
    which, make = CASES[name]
    b = make()
    step = max(b.n // 400, 1)
    sample = np.arange(0, b.n, step)
    (wave, used), (lane, none) = run(b, algo, second, 3, sample), run(b, algo, second, 2, sample)
    planned, claimed, *pairs = used
    assert none is None and claimed <= planned
    assert [planned, *pairs] == g.wave_tb_plan(b.qlen, b.tlen, g.device_info()["n_cu"]) or algo == g.LOCAL and not second
    assert pairs[which] > 0.9 * b.n, pairs
    assert_same(wave, lane, fields(algo, g.WITH_TB, second) + ["n_ops", "cigars"], "lane path")
    ref = O.align(b.subset(sample), algo, start_pos=g.WITH_TB, second_best=second, n_penalty=1)
    got = {f: v[sample] for f, v in wave.items() if isinstance(v, np.ndarray) and len(v) == b.n}
    got["cigars"] = wave["cigars"]
    assert_parity(got, ref, algo, g.WITH_TB, second)


def paths(b, scores=(1, 4, 6, 1), n_penalty=None, policy=3, **kw):
    g.lib().gasal2_set_dispatch(policy)
    a = g.Aligner(g.Parameters(**kw), int(b.qlen.max()), int(b.tlen.max()), b.n, scores=scores, n_penalty=n_penalty)
    try:
        a.run(b)
        return a.last_paths()
    finally:
        g.lib().gasal2_set_dispatch(0)
        a.close()


def test_packed_kernels_taken_and_left():
    short = related(7410, 300, (60, 200), (60, 300))
    long = related(7411, 4, (1200, 1200), (1200, 1200))   # H of 8400 at match 7
    strong = dict(scores=(7, 2, 3, 1))
    for algo, start in ((g.LOCAL, g.WITHOUT_START), (g.LOCAL, g.WITH_START), (g.GLOBAL, g.WITHOUT_START),
                        (g.SEMI_GLOBAL, g.WITHOUT_START), (g.SEMI_GLOBAL, g.WITH_START), (g.LOCAL, g.WITH_TB),
                        (g.GLOBAL, g.WITH_TB)):
        assert paths(short, algo=algo, start_pos=start) & 8, (algo, start)
        assert not paths(short, algo=algo, start_pos=start, policy=2) & 8, (algo, start)
    assert not paths(long, algo=g.LOCAL, start_pos=g.WITH_TB, **strong) & 8
    assert paths(short, algo=g.BANDED, k_band=32) & 32
    assert not paths(long, algo=g.BANDED, k_band=32, **strong) & 32
    assert paths(short, algo=g.KSW) & 16
    assert not paths(long, algo=g.KSW, **strong) & 16
    nn = g.make_batch([b"N" * 600, b"ACGT"], [b"N" * 600, b"ACGT"], seeds=np.array([3, 3], np.uint32))
    assert paths(nn, algo=g.KSW, n_penalty=1) & 16
    assert not paths(nn, algo=g.KSW, n_penalty=-7) & 16


@pytest.mark.parametrize("n,lq,lt,packed", [(64, 60, 2000, False), (64, 150, 150, True), (10_000, 8, 8, True)])
def test_few_local_pairs(n, lq, lt, packed):
    """LOCAL WITH_TB of few pairs: one-wave blocks for short queries against long targets, else this path."""
    b = related(7420 + n, n, (lq, lq), (lt, lt))
    assert bool(paths(b, algo=g.LOCAL, start_pos=g.WITH_TB, policy=0) & 8) == packed
