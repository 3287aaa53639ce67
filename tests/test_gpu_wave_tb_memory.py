"""Device memory of WITH_TB on the packed one-wave path: what a batch of unlike
lengths takes beside its CIGAR slots, and that the results stay those of the
lane kernels there."""
import numpy as np
import pytest
import torch

import gasal2_amd as g
from parity import assert_same, fields

pytestmark = pytest.mark.gpu


def run(b, algo, second, policy):
    """Results, device bytes the storage's batch took beside its CIGAR slots, and the paths."""
    g.lib().gasal2_set_dispatch(policy)
    a = g.Aligner(g.Parameters(algo=algo, start_pos=g.WITH_TB, secondBest=g.TRUE if second else g.FALSE),
                  int(b.qlen.max()), int(b.tlen.max()), b.n)
    try:
        a.load(b, per_pair=False)
        free = torch.cuda.mem_get_info()[0]
        a.run_resident()
        a.sync()
        took = free - torch.cuda.mem_get_info()[0] - a.result_views()[5] * b.n * 9 // 8
        out = a.download()
        out["cigars"] = [a.cigar(k) for k in range(0, b.n, max(b.n // 200, 1))]
        return out, took, a.last_paths()
    finally:
        g.lib().gasal2_set_dispatch(0)
        a.close()


def short_pairs_and_one(n, long_target):
    rng = np.random.default_rng(8100)
    base = rng.choice(list(b"ACGT"), long_target).astype(np.uint8)
    qs = [base[o:o + 40].tobytes() for o in rng.integers(0, 1000, n)]
    ts = [q[:20] + b"AC" + q[20:] + b"GATTACA" for q in qs]
    ts[n // 2] = base.tobytes()
    return g.make_batch(qs, ts)


def test_strip_records_of_one_long_target():
    """Second best keeps a record per strip of the batch: 40,000 pairs of 6
    strips and one of 12,500 take 1 MB, not 40,001 rows of 12,500 (2 GB)."""
    b = short_pairs_and_one(40_000, 100_000)
    got, took, paths = run(b, g.LOCAL, True, 3)
    assert paths & 6 == 6
    # checkpoints: 2500 waves of 12 iterations and 98 passes of 260 (8 KiB
    # each); fallback words, packed words and the rest below 300 MB
    assert took < (2500 * 12 + 98 * 260) * 8192 * 9 / 8 + 3e8, took
    lane, _, _ = run(b, g.LOCAL, True, 2)
    assert_same(got, lane, fields(g.LOCAL, g.WITH_TB, True) + ["n_ops", "cigars"], "lane path")


@pytest.mark.parametrize("algo,second", [(g.LOCAL, False), (g.LOCAL, True), (g.GLOBAL, False)])
def test_tile_budget_holds_for_short_queries(algo, second):
    """A pass lasts at least as many iterations as the group has lanes: 200
    queries of 20 bases against 14,000 want 400 MB of checkpoints and more for
    34 MB of tiles.  Over the budget the lane kernels run."""
    rng = np.random.default_rng(8200)
    t = rng.choice(list(b"ACGT"), 14_000).astype(np.uint8)
    b = g.make_batch([t[o:o + 20].tobytes() for o in rng.integers(0, 13_000, 200)], [t.tobytes()] * 200)
    budget = 100_000_000
    g.lib().gasal2_set_tile_budget(budget)
    try:
        got, took, _ = run(b, algo, second, 3)
    finally:
        g.lib().gasal2_set_tile_budget(64 << 30)
    assert took < budget * 9 / 8 + 1.5e8, took
    lane, _, _ = run(b, algo, second, 2)
    assert_same(got, lane, fields(algo, g.WITH_TB, second) + ["n_ops", "cigars"], "lane path")
