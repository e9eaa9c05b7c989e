"""bench.py times and reports the tile that sf_phys_substep_fused takes by itself."""
from __future__ import annotations

import pytest

import bench
from sailfish_amd import _lib


@pytest.mark.parametrize("prec,szI,szJ,named,tile", [
    (_lib.SF_FP64, 2048, 1024, 0, [64, 8]), (_lib.SF_FP32, 2048, 1024, 0, [64, 8]), (_lib.SF_FP64, 128, 64, 0, [16, 8]),
    (_lib.SF_FP64, 512, 256, 0, [32, 8]), (_lib.SF_FP64, 513, 255, 0, [64, 4]), (_lib.SF_FP64, 128, 64, 4, [64, 4])])
def test_reported_tile(prec, szI, szJ, named, tile):
    assert bench.phys_tile(prec, szI, szJ, named) == tile
