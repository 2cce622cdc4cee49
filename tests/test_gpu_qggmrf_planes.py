"""The qGGMRF prior at every number of planes a workgroup marches."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(3, 3, 3), (4, 16, 32), (18, 15, 33), (19, 17, 200), (35, 45, 95), (40, 72, 181),
                                  (67, 100, 130), (130, 100, 150)])
def test_qggmrf_planes_match_oracle(ctx, orc, dims):
    """One plane per workgroup (the smallest volumes) to sixteen, with ragged last chunks and
    tiles.  The 26 terms are summed in the oracle's order in float; what may differ is the last
    bit of a power, so a term's error is within 2^-23 of it and the sum's within 26 of those."""
    import lamino_amd as la

    say("qggmrf", dims)
    rng = np.random.default_rng(11)
    x = rng.standard_normal(dims).astype(np.float32)
    x[:, : dims[1] // 2] = 0.25  # flat part: zero differences
    g = np.zeros(dims, np.float32)
    want = orc.qggmrf(g, x, 1000.0, 1.2, prec=32)
    got = la.qggmrf(g.copy(), x, 1000.0, 1.2)
    assert np.max(np.abs(got - want)) <= 27 * 2**-23 * np.max(np.abs(want))
