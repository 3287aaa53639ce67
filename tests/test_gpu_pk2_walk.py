"""LOCAL WITH_TB two pairs a lane where the one-pair kernel's position encoding
does not fit (h, strip and column in 31 bits) and the packed kernel's does: the walk
reads the checkpoints of the kernel that ran."""
import numpy as np
import pytest

import gasal2_amd as g
from parity import assert_parity, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("length", [72, 136, 264, 520, 584])
def test_strong_matches(length, second):
    rng = np.random.default_rng(9700 + length)
    qs, ts = [], []
    for k in range(70):
        q = rng.choice(list(b"ACGT"), length - k % 9).astype(np.uint8)
        t = q.copy()
        t[rng.random(len(t)) < 0.03] = ord("G")
        qs.append(q.tobytes())
        ts.append(np.concatenate([t[:30], t[30 + k % 3:]]).tobytes())
    g.lib().gasal2_set_dispatch(2)
    try:
        b = g.make_batch(qs, ts)
        got, ref = run_both(b, g.LOCAL, g.WITH_TB, second, scores=(7, 8, 6, 1))
    finally:
        g.lib().gasal2_set_dispatch(0)
    assert_parity(got, ref, g.LOCAL, g.WITH_TB, second, b)
