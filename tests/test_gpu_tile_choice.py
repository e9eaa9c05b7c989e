"""The fused physics substep without a named tile: never much slower than with a 64-wide tile
named, on grids of about 250 to 800 32 x 8 tiles in both precisions, and the same results on
both sides of each line of the choice (as test_gpu_phys_tiles)."""
from __future__ import annotations

import sys

import pytest

from sailfish_amd import configs
from tests.test_gpu_phys_tiles import test_default_tile_matches_four_launches as matches_four_launches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("szI,szJ", [(512, 128), (416, 160), (352, 192), (480, 248), (544, 240), (544, 256), (672, 248), (768, 256),
                                     (256, 776)])
def test_choice_matches_four_launches(szI, szJ):
    matches_four_launches(szI, szJ)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("szI,szJ", [(352, 184), (512, 256), (475, 245), (513, 255), (704, 176), (640, 272), (768, 256),
                                     (640, 320)])
def test_choice_is_not_slower(szI, szJ, dt):
    """Within 10 % of the better of 64 x 4 and 64 x 8 (measured 0.72 to 1.03); 32 x 8 tiles up to
    576 of them took up to 1.22."""
    import torch
    from sailfish_amd.model2d import build_model
    from sailfish_amd.phys2d import PhysStepper, run_phys
    print(f"[case] tile choice {szI}x{szJ} {dt}", file=sys.stderr, flush=True)
    cfg = configs.random_smooth(szI, szJ, seed=3)
    cfg["dtfast"] = 1.0
    runs = []
    for tj in (0, 4, 8):
        ct, GRID, OCEAN, _B = build_model(cfg, dtype=torch.float64 if dt == "f64" else torch.float32, ndtfast=30)
        st = PhysStepper(GRID, OCEAN, tile_j=tj)
        g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            run_phys(ct, GRID, OCEAN, 30, st)
            with torch.cuda.graph(g, stream=s):
                run_phys(ct, GRID, OCEAN, 30, st, start_first=False)
        torch.cuda.synchronize()
        runs.append((g, (ct, GRID, OCEAN, st), []))
    for _ in range(11):
        for g, _keep, t in runs:
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            g.replay()
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
    auto, four, eight = (sorted(t)[5] for _g, _k, t in runs)
    print(f"[tile choice] {szI}x{szJ} {dt} {auto / min(four, eight):.3f}", file=sys.stderr, flush=True)
    assert auto < 1.1 * min(four, eight), (auto, four, eight)
