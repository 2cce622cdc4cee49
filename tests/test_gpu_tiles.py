"""The tiled spreader and interpolator at the sizes where its cutting can go wrong: fine grids
shorter than a block, tiles that do not divide the axis, every kernel width, rows cut between
jobs, and a record budget of one job, for shared-tilt grids (row slots) and for grids whose
tilt varies (first-cell slots)."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _tol(eps):
    """The kernel of width W = ceil(-log10(eps / 10)), made even, is accurate to about 10^(1 - W);
    a factor 10 above that, and not below the FP32 sums' 1e-5."""
    w = int(np.ceil(-np.log10(eps / 10)))
    w += w % 2
    return max(1e-5, 10.0 ** (2 - max(4, min(12, w))))


CASES = [((3, 2, 4), 5, 7, 3, 1e-5), ((13, 5, 7), 9, 10, 6, 1e-5), ((48, 6, 40), 20, 24, 9, 1e-5),
         ((10, 6, 14), 12, 13, 8, 1e-3), ((10, 6, 14), 12, 13, 8, 1e-6), ((10, 6, 14), 13, 12, 8, 1e-8),
         ((10, 6, 14), 13, 13, 8, 1e-10), ((21, 9, 23), 31, 33, 150, 1e-5), ((21, 9, 23), 31, 33, 400, 1e-5)]


@pytest.mark.parametrize("varying", [False, True])
@pytest.mark.parametrize("dims,R,C,P,eps", CASES)
def test_projectors_over_tile_edges(dims, R, C, P, eps, varying):
    import lamino_amd as la
    import oracle as orc

    say("tiles", dims, R, C, P, eps, varying)
    rng = np.random.default_rng(17)
    al = np.linspace(0.05, 3.0, P) if varying else np.full(P, np.radians(-33.0))
    ga = np.full(P, 0.4) if varying else 0.2 + 2 * np.pi * np.arange(P) / P
    pg = la.PolarGrid.per_projection(al, ga, R, C)
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    a = la.adjoint(p, pg, dims, eps=eps)
    assert _rel(a, orc.adjoint(p, dims, al, ga, eps=1e-12)) < _tol(eps)
    m = rng.standard_normal((3,) + dims).astype(np.float32)
    assert _rel(la.forward(m, pg, eps=eps), orc.forward(m, al, ga, R, C, eps=1e-12)) < _tol(eps)


@pytest.mark.parametrize("varying", [False, True])
def test_one_job_record_budget_changes_only_the_summation_order(monkeypatch, varying):
    import lamino_amd as la

    dims, R, C, P = (21, 9, 23), 31, 33, 150
    rng = np.random.default_rng(18)
    al = np.linspace(0.05, 3.0, P) if varying else np.full(P, np.radians(33.0))
    pg = la.PolarGrid.per_projection(al, 0.2 + 2 * np.pi * np.arange(P) / P, R, C)
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    whole = la.adjoint(p, pg, dims)
    monkeypatch.setenv("LAMINO_NUFFT_SLAB_BYTES", "1")
    # sums of at most a few thousand FP32 terms in another order
    assert _rel(la.adjoint(p, pg, dims), whole) < 1e-5
