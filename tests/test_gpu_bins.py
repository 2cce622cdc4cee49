"""The sorted point bins where a bucket is too large to be ranked whole, and at its edge."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("varying", [False, True])
@pytest.mark.parametrize("dims,R,C,P", [((3, 2, 4), 5, 7, 16), ((9, 6, 9), 16, 16, 1), ((9, 6, 9), 16, 17, 2),
                                        ((21, 9, 23), 31, 33, 300), ((4, 3, 5), 61, 61, 150)])
def test_projections_from_large_buckets(dims, R, C, P, varying):
    """Kernel width 8: the binned interpolators.  The order of the points in a bucket is fixed, so
    two grids built alike give the same bits, and the width's accuracy (about 10^(1 - 8), a factor
    10 above that and not below the FP32 sums' 1e-5) holds against the oracle."""
    import lamino_amd as la
    import oracle as orc

    say("bins", dims, R, C, P, varying)
    rng = np.random.default_rng(23)
    al = np.linspace(0.05, 3.0, P) if varying else np.full(P, np.radians(-33.0))
    ga = np.full(P, 0.4) if varying else 0.2 + 2 * np.pi * np.arange(P) / P
    m = rng.standard_normal((3,) + dims).astype(np.float32)
    one, two = (la.forward(m, la.PolarGrid.per_projection(al, ga, R, C), eps=1e-7) for _ in range(2))
    assert np.array_equal(one, two)
    want = orc.forward(m, al, ga, R, C, eps=1e-12)
    assert np.linalg.norm(one - want) <= 1e-5 * np.linalg.norm(want)
