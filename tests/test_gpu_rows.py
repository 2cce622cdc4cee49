"""The row-factorised spreader (MBIR1's and MBIR2's backprojection) and interpolator (forwards at
kernel widths above 6), which the default projectors at width 6 do not reach."""
import ctypes

import numpy as np
import pytest

from conftest import rel, say

pytestmark = pytest.mark.gpu

EPS = {4: 1e-3, 6: 1e-5, 8: 1e-6, 10: 1e-8, 12: 1e-10}


def _tol(w):
    """A kernel of width w is accurate to about 10^(1 - w); a factor 10 above that, and not below
    the FP32 sums' 1e-5."""
    return max(1e-5, 10.0 ** (2 - w))


def _ran(ctx, call, scopes):
    """call()'s result, and how often each timed scope ran in it."""
    from lamino_amd._lib import check

    check(ctx.lib.lam_timing_enable(ctx.h, 1))
    out = call()
    ms, n, got = ctypes.c_double(), ctypes.c_int64(), {}
    for s in scopes:
        check(ctx.lib.lam_timing_query(ctx.h, s.encode(), ctypes.byref(ms), ctypes.byref(n)))
        got[s] = n.value
    check(ctx.lib.lam_timing_enable(ctx.h, 0))
    return out, got


TILTS = [(30.0, None), (30.0, "1"), (30.0, "100000"), (-25.0, None), (-25.0, "1"), (90.0, None), (0.0, "1")]


@pytest.mark.parametrize("w", sorted(EPS))
@pytest.mark.parametrize("tilt,slab", TILTS)
def test_row_spreader(ctx, orc, monkeypatch, tilt, slab, w):
    """Both orders of the rows' first y cells, rows spanning the whole y period (90 degrees), all
    rows on one y cell (0 degrees); one row per group, several, and all in one."""
    import lamino_amd as la

    dims, R, C, P = (9, 5, 11), 13, 15, 7
    monkeypatch.setenv("LAMINO_NUFFT_ROWS", "spread")
    if slab:
        monkeypatch.setenv("LAMINO_NUFFT_SLAB_BYTES", slab)
    rng = np.random.default_rng(123)
    al, ga = np.full(P, np.radians(tilt)), np.linspace(0, 2 * np.pi, P, endpoint=False) + 0.4
    pg = la.PolarGrid.per_projection(al, ga, R, C)
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    a, ran = _ran(ctx, lambda: la.adjoint(p, pg, dims, eps=EPS[w]), ["spread_rows2d", "y_expand", "tile_spread"])
    assert ran["spread_rows2d"] > 0 and ran["y_expand"] > 0 and ran["tile_spread"] == 0, ran
    if slab == "1":
        assert ran["spread_rows2d"] == 7, ran   # half of the 13 rows, one per group
    e = rel(a, orc.adjoint(p, dims, al, ga, eps=1e-12))
    say(f"rows w {w} tilt {tilt} slab {slab}: adjoint rel {e:.2e}")
    assert e < _tol(w)


@pytest.mark.parametrize("w", [8, 10, 12])
@pytest.mark.parametrize("tilt,slab", TILTS)
def test_row_interpolator(ctx, orc, monkeypatch, tilt, slab, w):
    import lamino_amd as la

    dims, R, C, P = (9, 5, 11), 13, 15, 7
    if slab:
        monkeypatch.setenv("LAMINO_NUFFT_SLAB_BYTES", slab)
    rng = np.random.default_rng(124)
    al, ga = np.full(P, np.radians(tilt)), np.linspace(0, 2 * np.pi, P, endpoint=False) + 0.4
    pg = la.PolarGrid.per_projection(al, ga, R, C)
    m = rng.standard_normal((3,) + dims).astype(np.float32)
    y, ran = _ran(ctx, lambda: la.forward(m, pg, eps=EPS[w]), ["interp_rows2d", "y_contract", "tile_interp"])
    assert ran["interp_rows2d"] > 0 and ran["y_contract"] > 0 and ran["tile_interp"] == 0, ran
    if slab == "1":
        assert ran["interp_rows2d"] == 7, ran
    e = rel(y, orc.forward(m, al, ga, R, C, eps=1e-12))
    say(f"rows w {w} tilt {tilt} slab {slab}: forward rel {e:.2e}")
    assert e < _tol(w)


@pytest.mark.parametrize("eps", [1e-5, 1e-6])
def test_tuned_row_tiling_keeps_parity(ctx, orc, monkeypatch, eps):
    """The kernels that read the tuner's choice, before and after it: another tiling changes only
    the FP32 summation order.  Shapes that no other test tunes."""
    import lamino_amd as la

    dims, R, C, P = (87, 19, 85), 87, 83, 24
    monkeypatch.setenv("LAMINO_NUFFT_ROWS", "spread")
    rng = np.random.default_rng(67)
    al, ga = np.full(P, np.radians(30.0)), 2 * np.pi * np.arange(P) / P
    pg = la.PolarGrid.per_projection(al, ga, R, C)
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    m = rng.standard_normal((3,) + dims).astype(np.float32)
    a0, y0 = la.adjoint(p, pg, dims, eps=eps), la.forward(m, pg, eps=eps)
    T, ms = la.autotune_bins(pg, dims, eps=eps)
    a1, y1 = la.adjoint(p, pg, dims, eps=eps), la.forward(m, pg, eps=eps)
    say("tuned", T, f"{ms:.3f} ms", rel(a1, a0), rel(y1, y0))
    assert ms > 0 and T[0] >= 2 and T[2] >= 2
    assert rel(a1, a0) < 1e-5 and rel(y1, y0) < 1e-5
    assert rel(a1, orc.adjoint(p, dims, al, ga, eps=1e-12)) < 1e-4


@pytest.mark.parametrize("dims,R,C,P,eps,tilt,tiles", [((60, 60, 60), 17, 40, 20, 1e-5, 60.0, False), ((60, 60, 60), 17, 40, 20, 1e-5, 0.0, True),
                                                       ((31, 31, 31), 17, 40, 20, 1e-5, 60.0, True), ((48, 40, 60), 41, 43, 2, 1e-6, 90.0, False),
                                                       ((48, 40, 60), 41, 43, 2, 1e-8, 35.0, True), ((48, 12, 60), 41, 43, 60, 1e-6, 35.0, True)])
def test_adjoints_on_both_sides_of_the_line(ctx, orc, dims, R, C, P, eps, tilt, tiles):
    """Few rows against the planes they span go by rows, the others by tiles; one grid adds into
    what the other left."""
    import lamino_amd as la

    rng = np.random.default_rng(125)
    al, ga = np.full(P, np.radians(tilt)), 0.4 + 2 * np.pi * np.arange(P) / P
    pg = la.PolarGrid.per_projection(al, ga, R, C)
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    a, ran = _ran(ctx, lambda: la.adjoint(p, pg, dims, eps=eps), ["spread_rows2d", "tile_spread"])
    assert (ran["tile_spread"] > 0) == tiles and (ran["spread_rows2d"] > 0) == (not tiles), ran
    w = {v: k for k, v in EPS.items()}[eps]
    assert rel(a, orc.adjoint(p, dims, al, ga, eps=1e-12)) < _tol(w)
    assert rel(la.adjoint_multi([p, p], [pg, pg], dims, eps=eps), 2 * a) < 1e-5
