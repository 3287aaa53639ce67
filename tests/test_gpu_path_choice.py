"""Which kernels the automatic policy takes where one side clearly wins, by the
bits of gasal2_last_paths, the results equal to those of the other side."""
import numpy as np
import pytest
import torch

import gasal2_amd as g
from parity import assert_same, fields
from test_gpu_wave_tb_walk import related, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,length,packed", [(20_000, 16, False), (70_000, 24, False), (300, 200, True)])
def test_global_tb_of_short_pairs_on_lanes(n, length, packed):
    """A pass of the packed path lasts five iterations and the host plans every
    pair: 600,000 pairs of 16 x 16 bases 0.4 ms on lanes, 2.9 there."""
    b = related(7500 + n, n, (length, length), (length, length))
    sample = range(0, n, max(n // 100, 1))
    (auto, paths), (other, _) = run(b, g.GLOBAL, False, 0, sample), run(b, g.GLOBAL, False, 2 if packed else 3, sample)
    assert bool(paths & 4) == packed
    assert_same(auto, other, fields(g.GLOBAL, g.WITH_TB, False) + ["n_ops", "cigars"], "other side")


@pytest.mark.parametrize("start", [g.WITHOUT_START, g.WITH_START])
def test_packed_scores_take_no_panels(start):
    """The lane kernels' sequence panels are a row of the longest target's words for
    every pair (2 GB here); the packed path reads its pairs' own words."""
    rng = np.random.default_rng(7600)
    t = rng.choice(list(b"ACGT"), 100_000).astype(np.uint8)
    qs = [t[o:o + 40].tobytes() for o in rng.integers(0, 1000, 40_000)]
    b = g.make_batch(qs, qs[:-1] + [t.tobytes()])
    g.lib().gasal2_set_dispatch(3)
    a = g.Aligner(g.Parameters(algo=g.LOCAL, start_pos=start), 40, 100_000, b.n)
    try:
        a.load(b, per_pair=False)
        free = torch.cuda.mem_get_info()[0]
        a.run_resident()
        a.sync()
        took = free - torch.cuda.mem_get_info()[0]
        assert a.last_paths() & 8
        assert (a.download()["score"][:-1] == 40).all()
    finally:
        g.lib().gasal2_set_dispatch(0)
        a.close()
    assert took < 3e8, took


@pytest.mark.parametrize("n,lq,lt", [(1, 8, 8), (3000, 16, 16), (2000, 300, 30), (40, 1500, 1500)])
def test_few_scores_on_the_packed_path(n, lq, lt):
    """Few pairs LOCAL, scores and ends: the one-wave blocks, the other side, are slower at every shape."""
    b = related(7700 + n, n, (lq, lq), (lt, lt))
    out = []
    for policy in (0, 2):
        g.lib().gasal2_set_dispatch(policy)
        a = g.Aligner(g.Parameters(algo=g.LOCAL), lq, lt, n)
        try:
            out.append(a.run(b, per_pair=False))
            assert bool(a.last_paths() & 8) == (policy == 0)
        finally:
            g.lib().gasal2_set_dispatch(0)
            a.close()
    assert_same(out[0], out[1], fields(g.LOCAL, g.WITHOUT_START, False), "lane path")
