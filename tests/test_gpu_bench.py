"""The benchmark's own arithmetic on a small configuration."""
import importlib.util
import os

import pytest

from conftest import say

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("config", [1, 2])
def test_roofline_models_the_kernels_that_run(ctx, config):
    """Every kernel of the projectors has its own scope, and no model counts more work than the
    hardware can do in the time measured."""
    import lamino_amd as la
    from lamino_amd import synth

    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    pr = bench.Projectors(la, synth.config(config))
    ms, spread_ms, spread_cnt = pr.timed(3, 1)
    kernels = pr.diagnostic(2)
    roof = bench.roofline(pr, kernels, spread_ms, spread_cnt, bench.WORKLOAD_KEY[config])
    say(roof)
    assert {"spread", "tile_spread", "tile_merge", "interp", "tile_interp"} <= set(kernels)
    assert kernels["tile_spread"]["total_ms"] + kernels["tile_merge"]["total_ms"] <= 1.1 * kernels["spread"]["total_ms"]
    assert {"tile_spread", "tile_interp"} <= set(roof["binding"])
    assert all(0 < b["frac"] <= 1 for b in [roof, *roof["binding"].values()]), roof
    pr.release()
