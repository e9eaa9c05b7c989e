"""The tracer step with one buffer for both new tracers, as when each was stepped and copied
back by itself: the same bits as with two."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests.helpers2d import bitwise_equal
from tests.test_gpu_baroclinic import _cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_shared_new_buffer(dt):
    import torch
    from sailfish_amd.baroclinic import Tracers
    from sailfish_amd.main3d import initial_depths
    from sailfish_amd.model2d import build_model3d
    print(f"[case] shared tracer buffer {dt}", file=sys.stderr, flush=True)
    szI, szJ, N = 67, 19, 7
    _ct, GRID, OCEAN, _B = build_model3d(_cfg(szI, szJ, N, seed=1), N=N, ndtfast=6, dt=12.0,
                                         dtype=torch.float64 if dt == "f64" else torch.float32)
    initial_depths(GRID, OCEAN)
    rng = np.random.default_rng(2)
    for t in (OCEAN.Huon, OCEAN.Hvom):
        t.copy_(torch.from_numpy(40.0 * rng.standard_normal(t.shape)))
    T, S = 10.0 + rng.random((N, szJ, szI)), 35.0 + rng.standard_normal((N, szJ, szI))
    out = []
    for shared in (False, True):
        tr = Tracers(GRID, OCEAN, T=T, S=S)
        tr.Hz_old.copy_(GRID.Hz)
        if shared:
            tr.S_new = tr.T_new
        for _ in range(3):
            tr.step(GRID, OCEAN, 60.0)
        torch.cuda.synchronize()
        out.append([t.cpu().numpy() for t in (tr.T, tr.S)])
    for a, b in zip(*out):
        assert bitwise_equal(a, b)
