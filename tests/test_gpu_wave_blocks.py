"""The packed one-wave path's score modes on batches of equal pairs on each side of
what its blocks of four waves take: a device's worth of pairs (four a compute
unit), targets of more than one pass, queries of at least a pass's columns."""
import numpy as np
import pytest

import gasal2_amd as g
from test_gpu_wave import MODES, both_paths

pytestmark = pytest.mark.gpu


def equal_pairs(n, lq, lt):
    rng = np.random.default_rng(3700 + n + lq)
    base = rng.choice(list(b"ACGT"), 1 << 14).astype(np.uint8)
    qs, ts = [], []
    for o, at in zip(rng.integers(0, 1 << 13, n), rng.integers(0, max(lt - lq, 1), n)):
        t = base[o:o + lt]
        q = t[at:at + lq].copy()
        q[rng.random(lq) < 0.05] = ord("T")
        qs.append(q.tobytes())
        ts.append(t.tobytes())
    return g.make_batch(qs, ts)


@pytest.mark.parametrize("per_cu", [4, 5])
@pytest.mark.parametrize("lq,lt", [(121, 1033), (40, 1100)])
@pytest.mark.parametrize("algo,start", MODES)
def test_equal_pairs(algo, start, lq, lt, per_cu):
    both_paths(equal_pairs(per_cu * g.device_info()["n_cu"] + per_cu % 4, lq, lt), algo, start)
