"""FFT passes at the edges of their tiles: lines per workgroup that do not divide its threads,
partial last tiles, lines shorter than a load batch and longer than a wave."""
import numpy as np
import pytest

from conftest import rel, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 2, 1), (1, 1, 2), (3, 2, 47), (2, 3, 49), (1, 180, 35), (5, 90, 129), (129, 4, 5),
                                   (33, 5, 64), (2, 65, 256), (1, 256, 513), (7, 205, 50), (2, 53, 100), (1, 12, 3840),
                                   (1, 3840, 2), (800, 6, 10)])
@pytest.mark.parametrize("shifted", [False, True])
def test_fft2_at_tile_edges(ctx, orc, shape, shifted):
    """Both axes' passes against a transform in 64 bits.  The bound is a single-precision
    transform's: each of log2(n) stages adds about one rounding (2^-24) of relative L2 error per
    element, six times that where a convolution (three transforms) stands for the line."""
    import lamino_amd as la

    say("fft2 lines", shape, shifted)
    rng = np.random.default_rng(7)
    x = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    x64 = x.astype(np.complex128)
    want = orc.shift2(np.fft.fft2(orc.shift2(x64, inverse=False)), inverse=True) if shifted else np.fft.fft2(x64)
    assert rel(la.fft2(x, -1, shifted=shifted), want) < 6 * 2**-24 * (1 + np.log2(shape[1] * shape[2]))


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 8, 9, 13, 15, 16, 17, 23, 31, 32, 33, 34, 41, 63, 64, 65])
@pytest.mark.parametrize("planes,rows", [(1, 5), (3, 37), (7, 130)])
def test_short_contiguous_lines(ctx, orc, planes, rows, n):
    """Lines of up to 32 points share a wave, eight to thirty-two lanes each; one longer and the
    last partial tile.  The bound is that of the test above."""
    import lamino_amd as la

    say("short lines", planes, rows, n)
    rng = np.random.default_rng(8)
    x = (rng.standard_normal((planes, rows, n)) + 1j * rng.standard_normal((planes, rows, n))).astype(np.complex64)
    assert rel(la.fft2(x, -1), np.fft.fft2(x.astype(np.complex128))) < 6 * 2**-24 * (1 + np.log2(rows * n))
