"""GPU parity of WITH_TB on the packed one-wave path (4, 16 or 64 lanes per
pair, tiles rebuilt from its checkpoints), bit-exact against the oracle and the
lane kernels: scores, ends, starts, second best and CIGARs.  Shapes cross the
path's edges: strips on each side of a pass (8, 32 and 128 strips), queries of
fewer words than a group has lanes, single bases, pairs of unlike size in one
wave; repeats give ties and second bests that many strips could hold."""
import numpy as np
import pytest

import gasal2_amd as g
from parity import assert_parity, assert_same, fields, run_both
from test_gpu_wave import edge_batch

pytestmark = pytest.mark.gpu

MODES = [(g.LOCAL, False), (g.LOCAL, True), (g.GLOBAL, False)]


def both_paths(b, algo, second, **kw):
    """The batch on the one-wave path, then one or two pairs per lane."""
    runs = []
    for policy in (3, 2):
        g.lib().gasal2_set_dispatch(policy)
        try:
            got, ref = run_both(b, algo, g.WITH_TB, second, **kw)
        finally:
            g.lib().gasal2_set_dispatch(0)
        assert_parity(got, ref, algo, g.WITH_TB, second, b)
        runs.append(got)
    assert_same(runs[0], runs[1], fields(algo, g.WITH_TB, second) + ["n_ops", "cigars"], "lane path")


def pass_edges(seed):
    """Targets of 7 to 9, 31 to 33 and 127 to 129 strips, queries of 1 to 80 words."""
    rng = np.random.default_rng(seed)
    qs, ts = [], []
    for strips in (1, 7, 8, 9, 31, 32, 33, 127, 128, 129):
        for words in (1, 3, 4, 5, 6, 16, 17, 18, 80):
            lt, lq = 8 * strips - int(rng.integers(0, 8)), 8 * words - int(rng.integers(0, 8))
            t = rng.choice(list(b"ACGT"), lt).astype(np.uint8)
            q = rng.choice(list(b"ACGT"), lq).astype(np.uint8)
            m = min(lq, lt)
            o = int(rng.integers(0, lt - m + 1))
            q[:m] = t[o:o + m]
            q[rng.random(lq) < 0.05] = ord("C")
            if lq > 30:   # an indel
                q = np.concatenate([q[:20], q[23:], q[:3]])
            qs.append(q.tobytes())
            ts.append(t.tobytes())
    return g.make_batch(qs, ts)


@pytest.mark.parametrize("scores", [(1, 4, 6, 1), (2, 3, 5, 2), (7, 8, 0, 1)])
@pytest.mark.parametrize("algo,second", MODES)
def test_edges(algo, second, scores):
    both_paths(edge_batch(4100 + scores[0]), algo, second, scores=scores, n_penalty=1)


@pytest.mark.parametrize("algo,second", MODES)
def test_pass_edges(algo, second):
    both_paths(pass_edges(4200), algo, second)


@pytest.mark.parametrize("n", [1, 3, 4, 15, 17, 700])
@pytest.mark.parametrize("algo,second", MODES)
def test_full_features(algo, second, n):
    both_paths(g.synth_batch(2, 4300 + n, n), algo, second, is_rc=True, n_penalty=1)


@pytest.mark.parametrize("algo,second", MODES)
def test_mixed_lengths(algo, second):
    both_paths(g.synth_batch(3, 4400, 90), algo, second)


def test_second_best_of_repeats():
    rng = np.random.default_rng(4500)
    units = [b"A", b"AC", b"ACG", b"ACGTTGCA", b"AAAAAAAC", b"ACGTN"]
    qs, ts = [], []
    for _ in range(400):
        u, v = (units[int(rng.integers(len(units)))] for _ in range(2))
        q = (u * 400)[:int(rng.integers(1, 200))]
        t = (v * 20)[:int(rng.integers(0, 60))] + (u * 400)[:int(rng.integers(1, 300))] + (v * 9)[:int(rng.integers(0, 60))]
        qs.append(q)
        ts.append(t)
    for scores in ((1, 4, 6, 1), (3, 1, 1, 1)):
        both_paths(g.make_batch(qs, ts), g.LOCAL, True, scores=scores, n_penalty=1)


@pytest.mark.parametrize("algo,second", MODES)
def test_no_score_tables(algo, second):
    """Nibbles that share a score-table class ('I' and 'A'): the lane kernels and
    the one-wave direction words run in the same buffer."""
    b = edge_batch(4600)
    q = bytearray(b.query(3))
    q[5:7] = b"IA"
    both_paths(g.make_batch([bytes(q)] + [b.query(i) for i in range(1, b.n)], [b.target(i) for i in range(b.n)]), algo, second)


@pytest.mark.parametrize("algo,second", MODES)
def test_long_pairs_on_four_waves(algo, second):
    """Targets of 2 to 9 passes of 128 strips, the block's waves with unlike numbers of them."""
    rng = np.random.default_rng(4700)
    qs, ts = [], []
    for lq, lt in ((2000, 2048), (2000, 2049), (1500, 4096), (1500, 4097), (3000, 5200), (900, 9100), (4000, 3100), (40, 4200)):
        t = rng.choice(list(b"ACGT"), lt).astype(np.uint8)
        q = rng.choice(list(b"ACGT"), lq).astype(np.uint8)
        m, o = min(lq, lt), max(lt - lq, 0) // 2
        q[:m] = t[o:o + m]
        q[rng.random(lq) < 0.08] = ord("G")
        q = np.delete(q, range(lq // 2, lq // 2 + 9))
        qs.append(q.tobytes())
        ts.append(t.tobytes())
    both_paths(g.make_batch(qs, ts), algo, second)
