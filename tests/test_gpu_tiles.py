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


def test_more_buckets_than_one_launch_has_waves(monkeypatch):
    """2^26 waves are more than a launch holds.  1024 row slots over 67,200 tiles (a wide, flat
    volume at kernel width 8) are 68.8 million buckets; the same call cut by first y cells has a
    million.  Both orders sum at most a few thousand FP32 terms per cell."""
    import lamino_amd as la

    dims, R, C, P = (672, 4, 672), 2048, 8, 2
    pg = la.PolarGrid.per_projection(np.full(P, np.radians(30.0)), np.array([0.3, 1.7]), R, C)
    p = np.random.default_rng(19).standard_normal((P, R, C)).astype(np.float32)
    say("many buckets")
    rows = la.adjoint(p, pg, dims, eps=1e-6)
    monkeypatch.setenv("LAMINO_NUFFT_ROWS", "0")
    assert _rel(rows, la.adjoint(p, pg, dims, eps=1e-6)) < 1e-5


def test_more_detector_lines_than_one_launch_has_waves():
    """65,500 projections (an FFT launch takes up to 65,535 planes) of 1026 half rows are more than
    2^26 lines, one wave each; the halves of the scan are below that, and their adjoints add up to the whole one's.  A job sums up to 5120 points
    one after another in FP32, and about 330 jobs are summed per cell: 4 sqrt(5450) 2^-24."""
    import lamino_amd as la

    dims, R, C, P = (9, 5, 11), 2052, 1, 65500
    ga = 2 * np.pi * np.arange(P) / P
    p = np.random.default_rng(20).standard_normal((P, R, C), dtype=np.float32)
    say("many lines")

    def back(a, b):
        pg = la.PolarGrid.per_projection(np.full(b - a, np.radians(30.0)), ga[a:b], R, C)
        return la.adjoint(p[a:b], pg, dims)

    assert _rel(back(0, P), back(0, P // 2) + back(P // 2, P)) < 4 * 5450**0.5 * 2**-24


@pytest.mark.parametrize("planes,rows", [(1, "1"), (40, "1"), (300, "1"), (40, "spread"), (300, "spread")])
def test_adjoint_over_the_record_budget_can_be_captured(monkeypatch, planes, rows):
    """Once its plan is there, an adjoint whose records (row slabs) exceed the budget, in groups of one
    job (row) and of several, only launches kernels: it can be captured, and each replay gives the
    eager call's bits for the input of the moment."""
    import ctypes

    import lamino_amd as la
    from lamino_amd._lib import check

    dims, R, C, P = (21, 9, 23), 31, 33, 150
    monkeypatch.setenv("LAMINO_NUFFT_SLAB_BYTES", str(4096 * planes))   # a record of width 6: 512 complex values
    monkeypatch.setenv("LAMINO_NUFFT_ROWS", rows)
    say("captured adjoint", planes, rows)
    ctx = la.Context()
    lib, stream = ctx.lib, ctypes.c_void_p(ctx.lib.lam_ctx_stream(ctx.h))
    pg = la.PolarGrid.per_projection(np.full(P, np.radians(33.0)), 0.2 + 2 * np.pi * np.arange(P) / P, R, C, ctx=ctx)
    proj, out = ctx.alloc((P, R, C)), ctx.alloc((3,) + dims)
    rng = np.random.default_rng(21)
    d = (ctypes.c_int64 * 3)(*dims)

    def call():
        check(lib.lam_adjoint(ctx.h, pg.h, d, 1e-5, ctypes.c_void_p(proj.ptr),
                              *[ctypes.c_void_p(q) for q in out.comps()]))

    def result():
        ctx.sync()
        got = out.download()
        out.zero()
        ctx.sync()
        return got

    proj.upload(rng.standard_normal((P, R, C)).astype(np.float32))
    call()
    ctx.sync()
    graph, launch = ctypes.c_void_p(), ctypes.c_void_p()
    assert lib.hipStreamBeginCapture(stream, 1) == 0   # this thread's calls
    try:
        call()
    finally:
        ended = lib.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert ended == 0
    assert lib.hipGraphInstantiate(ctypes.byref(launch), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        proj.upload(rng.standard_normal((P, R, C)).astype(np.float32))
        call()
        want = result()
        assert lib.hipGraphLaunch(launch, stream) == 0
        assert np.array_equal(result(), want) and np.linalg.norm(want) > 0
    ctx.sync()
    lib.hipGraphExecDestroy(launch)
    lib.hipGraphDestroy(graph)
    monkeypatch.delenv("LAMINO_NUFFT_SLAB_BYTES")
    call()
    assert _rel(result(), want) < 1e-5   # the same sums in another order


@pytest.mark.parametrize("dims,R,C,P", [((48, 6, 40), 11, 24, 5), ((48, 6, 40), 81, 24, 5), ((48, 6, 40), 141, 24, 5),
                                        ((64, 6, 64), 201, 16, 4), ((64, 6, 64), 201, 70, 3)])
def test_plans_scanned_in_one_workgroup_and_in_several(dims, R, C, P):
    """Counts of less than one block of 2048, of several in one workgroup (864 to 10,224 buckets),
    and of several workgroups (31,512); row slots below and above a wave's 64."""
    import lamino_amd as la
    import oracle as orc

    say("plan scans", dims, R, C, P)
    rng = np.random.default_rng(22)
    al, ga = np.full(P, np.radians(31.0)), 0.3 + 2 * np.pi * np.arange(P) / P
    pg = la.PolarGrid.per_projection(al, ga, R, C)
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    assert _rel(la.adjoint(p, pg, dims), orc.adjoint(p, dims, al, ga, eps=1e-12)) < _tol(1e-5)
    m = rng.standard_normal((3,) + dims).astype(np.float32)
    assert _rel(la.forward(m, pg), orc.forward(m, al, ga, R, C, eps=1e-12)) < _tol(1e-5)


@pytest.mark.parametrize("dims,R,C,P,eps,varying", [((9, 5, 11), 60, 60, 150, 1e-5, False), ((3, 3, 3), 60, 61, 100, 1e-5, False),
                                                    ((22, 22, 3), 149, 9, 150, 1e-8, False), ((5, 3, 3), 91, 31, 100, 1e-3, True),
                                                    ((20, 14, 15), 61, 61, 120, 1e-8, True)])
def test_tiles_with_many_jobs(dims, R, C, P, eps, varying):
    """Small volumes under many points: tiles of more than 24 jobs, whose jobs are longer."""
    import lamino_amd as la
    import oracle as orc

    say("deep tiles", dims, R, C, P, eps, varying)
    rng = np.random.default_rng(24)
    al = np.linspace(0.05, 3.0, P) if varying else np.full(P, np.radians(31.0))
    ga = np.full(P, 0.4) if varying else 0.3 + 2 * np.pi * np.arange(P) / P
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    a = la.adjoint(p, la.PolarGrid.per_projection(al, ga, R, C), dims, eps=eps)
    assert _rel(a, orc.adjoint(p, dims, al, ga, eps=1e-12)) < _tol(eps)


@pytest.mark.parametrize("dims,R,C,P,eps,tiles", [((9, 5, 11), 13, 15, 20, 1e-5, False), ((9, 5, 11), 13, 15, 21, 1e-5, True),
                                                  ((4, 4, 4), 61, 61, 40, 1e-3, False), ((4, 4, 4), 61, 61, 30, 1e-3, True),
                                                  ((4, 4, 4), 41, 31, 20, 1e-8, False), ((6, 5, 7), 41, 31, 20, 1e-10, True),
                                                  ((31, 9, 31), 45, 45, 60, 1e-6, True)])
def test_first_cell_grids_on_both_sides_of_the_line(ctx, dims, R, C, P, eps, tiles):
    """Grids of varying tilt: fewer than 2048 points, points crowded into a few tiles and wide
    kernels over fewer than six tiles go by 3-D bins; both against the oracle."""
    import ctypes

    import lamino_amd as la
    import oracle as orc
    from lamino_amd._lib import check

    say("first-cell line", dims, R, C, P, eps, tiles)
    rng = np.random.default_rng(25)
    al, ga = np.linspace(0.05, 3.0, P), np.full(P, 0.4)
    pg = la.PolarGrid.per_projection(al, ga, R, C)
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    check(ctx.lib.lam_timing_enable(ctx.h, 1))
    a = la.adjoint(p, pg, dims, eps=eps)
    ms, n = ctypes.c_double(), ctypes.c_int64()
    check(ctx.lib.lam_timing_query(ctx.h, b"tile_spread", ctypes.byref(ms), ctypes.byref(n)))
    check(ctx.lib.lam_timing_enable(ctx.h, 0))
    assert (n.value > 0) == tiles
    assert _rel(a, orc.adjoint(p, dims, al, ga, eps=1e-12)) < _tol(eps)
    acc = la.adjoint_multi([p, p], [pg, pg], dims, eps=eps)
    assert _rel(acc, 2 * a) < 1e-5   # the second grid adds into the first one's fine grid


@pytest.mark.parametrize("varying", [False, True])
@pytest.mark.parametrize("P", [255, 256, 257, 700, 2500])
def test_buckets_of_many_runs_keep_the_points_order(P, varying):
    """Up to 256 runs of a bucket are ranked by a wave, more by a workgroup.  The order of a bucket's
    points is theirs, so two plans give the same bits, and the sums are the oracle's."""
    import lamino_amd as la
    import oracle as orc

    dims, R, C = (9, 5, 11), 11, 13
    say("many runs", P, varying)
    rng = np.random.default_rng(26)
    al = np.linspace(0.05, 3.0, P) if varying else np.full(P, np.radians(31.0))
    ga = np.full(P, 0.4) if varying else 0.3 + 2 * np.pi * np.arange(P) / P
    p = rng.standard_normal((P, R, C)).astype(np.float32)
    one, two = (la.adjoint(p, la.PolarGrid.per_projection(al, ga, R, C), dims) for _ in range(2))
    assert np.array_equal(one, two)
    assert _rel(one, orc.adjoint(p, dims, al, ga, eps=1e-12)) < _tol(1e-5)
