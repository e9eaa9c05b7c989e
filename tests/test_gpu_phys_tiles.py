"""The tile the fused physics substep picks by itself on each grid size (tile_j = 0): core and
ring on different waves (16 x 8 and 32 x 8 tiles) on small grids, 64-wide tiles above.  Each
shape sits at an edge of the choice or of a tile (remainders 0, 1, 2; one tile more or less
than a CU count).  FP64 equals the four-launch form bit for bit; FP32 stays within 2e-6 of
each field's magnitude (the fused form contracts multiply-adds, ~1e-7 relative each)."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from sailfish_amd import configs
from tests.helpers2d import bitwise_equal

pytestmark = pytest.mark.gpu

NAMES = ("zeta", "ubar", "vbar", "rzeta", "rubar", "rvbar", "Zt_avg1", "DU_avg1", "DV_avg1")


def _same(A, B, exact):
    bad = []
    for n in NAMES:
        a, b = (getattr(x, n).cpu().numpy().astype(np.float64) for x in (A, B))
        ok = bitwise_equal(a, b) if exact else np.abs(a - b).max() <= 2e-6 * max(np.abs(b).max(), 1e-30)
        if not ok:
            bad.append((n, float(np.abs(a - b).max())))
    return bad


# 16 x 8 tiles: up to 256 of them; 32 x 8: up to 576; FP64 64 x 4: up to 768; then 64 x 8
SHAPES = [(4, 4), (17, 9), (18, 10), (33, 7), (256, 128), (257, 128), (49, 650), (512, 257), (576, 256), (577, 255),
          (513, 300), (640, 320), (705, 130), (1025, 385)]


@pytest.mark.parametrize("szI,szJ", SHAPES)
def test_default_tile_matches_four_launches(szI, szJ):
    import torch
    from sailfish_amd.model2d import build_model
    from sailfish_amd.phys2d import PhysStepper, run_phys
    cfg = configs.random_smooth(szI, szJ, seed=szI + 7 * szJ)
    cfg["dtfast"] = 1.0
    for dt in (torch.float64, torch.float32):
        print(f"[case] default tile {szI}x{szJ} {dt}", file=sys.stderr, flush=True)
        out = []
        for fused in (True, False):
            ct, GRID, OCEAN, _B = build_model(cfg, dtype=dt, ndtfast=30)
            run_phys(ct, GRID, OCEAN, 4, PhysStepper(GRID, OCEAN, fused=fused))
            out.append(OCEAN)
        bad = _same(*out, dt == torch.float64)
        assert not bad, bad


@pytest.mark.parametrize("szI,szJ", [(18, 10), (130, 66), (258, 130), (769, 384)])
def test_default_coupled_tile_matches_four_launches(szI, szJ):
    import torch
    from sailfish_amd.coupled3d import main3d_coupled
    from sailfish_amd.model2d import build_model3d
    cfg = configs.random_smooth(szI, szJ, seed=szI)
    cfg["dtfast"] = 1.0
    for dt in (torch.float64, torch.float32):
        print(f"[case] default coupled tile {szI}x{szJ} {dt}", file=sys.stderr, flush=True)
        out = []
        for fused in (True, False):
            ct, GRID, OCEAN, B = build_model3d(cfg, N=4, ndtfast=4, dt=4.0, dtype=dt)
            st = main3d_coupled(ct, GRID, OCEAN, B, 3, fused=fused)
            OCEAN.rzeta, OCEAN.rubar, OCEAN.rvbar = st.DU_avg2, st.DV_avg2, st.Fu[0]
            out.append(OCEAN)
        bad = _same(*out, dt == torch.float64)
        assert not bad, bad


@pytest.mark.parametrize("szI,szJ", [(33, 17), (66, 41), (512, 128), (513, 128)])
def test_default_closure_tile_matches_64x4(szI, szJ):
    """The closure's default tile (32 x 8 with its own ring waves up to one tile per CU) against
    64 x 4 tiles: the same network arithmetic per point, so both precisions bit for bit."""
    import torch
    from sailfish_amd.closure import ClosureMLP, Model
    cfg = configs.random_smooth(szI, szJ, seed=5)
    cfg["dtfast"] = 1.0
    mlp = ClosureMLP(seed=3)
    mlp.set_norm(np.zeros(45), np.ones(45), np.array([0.0, 1e-7, 0.0, 1e-7]))
    for dt in (torch.float64, torch.float32):
        print(f"[case] default closure tile {szI}x{szJ} {dt}", file=sys.stderr, flush=True)
        out = []
        for tj in (0, 4):
            m = Model(cfg, dt)
            m.stepper.tile_j = tj
            for _ in range(4):
                m.step(mlp)
            out.append(m.OCEAN)
        bad = _same(*out, True)
        assert not bad, bad
    mlp.close()
