"""Which kernels the automatic policy takes where one side clearly wins, by the
bits of gasal2_last_paths, the results equal to those of the other side."""
import pytest

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
