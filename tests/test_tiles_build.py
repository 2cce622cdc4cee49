"""Properties of the tile kernels that show in the compiler's output, not in a result."""
import os
import re
import subprocess

import pytest

from lamino_amd import build as recipe


@pytest.fixture(scope="module")
def tiles_ir():
    """Unoptimised LLVM IR of the device side of tiles.hip, as {function: body}."""
    cmd = [recipe.HIPCC, *recipe.COMMON_FLAGS, "-O0", "--offload-device-only", "-emit-llvm", "-S", "-o", "-",
           os.path.join(recipe.CSRC, "tiles.hip")]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return {m.group(1): m.group(2) for m in re.finditer(r"^define [^@]*@([\w.$]+)\(.*?\{\n(.*?)^\}", r.stdout, re.M | re.S)}


def test_staged_batches_are_ordered_between_lanes(tiles_ir):
    """The spreader's wave hands its points from lane to lane through LDS without a workgroup
    barrier.  The compiler has to keep three orders: the last batch's reads, the clear, the
    stamps and the next reads.  One fence between each, in all ten instantiations (five kernel
    widths, row and first-cell slots)."""
    fences = {f: len(re.findall(r'fence syncscope\("wavefront"\) acq_rel', b)) for f, b in tiles_ir.items()}
    staging = {f: n for f, n in fences.items() if "k_tile_spread" in f and n}
    assert len(staging) == 10 and set(staging.values()) == {3}, staging
