"""The open edges at the sizes where their workgroup's rounds of 1024 edge points end: below,
at and past one and two rounds, with edges closed in between and edges without outer values.
FP64 against the oracle, as the small grids: bit for bit without the volume constraint,
within 1e-12 of each field's maximum with it (the boundary sums run in another order)."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from sailfish_amd import configs
from tests.helpers2d import bitwise_equal
from tests.test_gpu_open import NAMES, _ext, _gpu, _oracle

pytestmark = pytest.mark.gpu


# edge points: 14, 1024, 1025 (north and west), 1466, 2198
@pytest.mark.parametrize("szI,szJ,flags", [(6, 5, 15), (502, 14, 15), (1004, 25, 1 | 8), (700, 37, 15),
                                           (1100, 4, 4 | 8 | 2)])
@pytest.mark.parametrize("volcons", [False, True])
def test_open_edges_rounds(szI, szJ, flags, volcons):
    import torch
    print(f"[case] open edge rounds {szI}x{szJ} flags={flags} volcons={volcons}", file=sys.stderr, flush=True)
    cfg = configs.random_smooth(szI, szJ, seed=szI + flags)
    ez, eu = _ext(szI, szJ, flags)
    ez[3], eu[0] = None, None
    ct, OCEAN = _gpu(cfg, torch.float64, flags, volcons, ez, eu, 4, dt=0.5)
    o = _oracle(cfg, ct, flags, volcons, ez, eu, 4, dt=0.5)
    bad = []
    for n in NAMES:
        for k in range(3):
            g = getattr(OCEAN, f"{n}_t{k}").detach().cpu().numpy()
            r = o.st.v(n, k)
            if volcons:
                if not np.abs(g - r).max() <= 1e-12 * max(np.abs(r).max(), 1e-30):
                    bad.append((n, k, float(np.abs(g - r).max() / max(np.abs(r).max(), 1e-30))))
            elif not bitwise_equal(g, r):
                bad.append((n, k))
    assert not bad, bad
