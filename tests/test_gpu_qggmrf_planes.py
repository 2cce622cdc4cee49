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


@pytest.mark.parametrize("p", [1.0, 1.2, 2.0, 2.5])
@pytest.mark.parametrize("scale", [1e-30, 1e-3, 1e4])
def test_qggmrf_powers_match_oracle(ctx, orc, p, scale):
    """The power of a difference over its range and the exponents' (2 - p positive, zero and
    negative), an infinite voxel among them: the same finite values within a last bit of each of
    the 26 terms, and the same values that are not finite."""
    import lamino_amd as la

    say("qggmrf powers", p, scale)
    rng = np.random.default_rng(12)
    x = (rng.standard_normal((7, 9, 14)) * scale).astype(np.float32)
    x[3, 4, 6] = np.inf
    g = np.zeros_like(x)
    with np.errstate(all="ignore"):
        want = orc.qggmrf(g, x, 2.0, p, prec=32)
    got = la.qggmrf(g.copy(), x, 2.0, p)
    ok = np.isfinite(want)
    assert np.array_equal(ok, np.isfinite(got)) and ok.sum() > ok.size // 2
    assert np.max(np.abs(got[ok] - want[ok])) <= 27 * 2**-23 * np.max(np.abs(want[ok]))
