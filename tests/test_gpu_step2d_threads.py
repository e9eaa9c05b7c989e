"""The fused barotropic substep on both sides of its thread-count rule (up to 256 tiles of
64 x 8 points: a thread per frame point; more: two points a thread), bit for bit in FP64
against the CPU oracle: full and ragged last tiles, shifted tile origins, tile counts that
do not divide by eight, copied velocity boundaries and masked interior columns."""
from __future__ import annotations

import sys

import pytest

from sailfish_amd import configs
from tests.helpers2d import compare_fused
from tests.test_gpu_step2d_fused import _run

pytestmark = pytest.mark.gpu

GRAD = {"ubar": ["GRA", "CLO", "GRA", "CLO"], "zeta": ["GRA", "CLO", "GRA", "CLO"]}


@pytest.mark.parametrize("szI,szJ,fix_q5,lbc,mode", [
    (512, 256, True, None, "main2d"),        # 256 tiles, none ragged
    (190, 688, True, None, "main2d"),        # 258
    (513, 257, True, None, "main3d"),        # 297, both origins shifted
    (521, 259, True, GRAD, "main2d"),        # 297, copies, ragged
    (1024, 256, False, None, "main3d"),      # 512, masked interior columns
    (1024, 256, False, GRAD, "main2d"),
    (321, 9, True, GRAD, "main3d"),          # 12, both origins shifted
])
def test_fused_fp64_bitwise_by_tiles(szI, szJ, fix_q5, lbc, mode):
    print(f"[case] fused tiles {mode} {szI}x{szJ} fix_q5={fix_q5} {lbc}", file=sys.stderr, flush=True)
    cfg = configs.random_smooth(szI, szJ, seed=szI + 7 * szJ)
    prod, orc = _run(cfg, 4 if mode == "main2d" else 1, mode, fix_q5, lbc=lbc)
    bad = compare_fused(prod, orc, szI, szJ, szI if fix_q5 else szJ)
    assert not bad, bad
