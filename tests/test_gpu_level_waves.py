"""set_maxflux and omega at the edges of their split over levels (four waves, each a run of a
quarter of the levels in batches of four; up to 64 levels for omega, deeper grids its
one-thread form): FP64, bit for bit against the reference's loops in NumPy."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from sailfish_amd import configs
from tests.helpers2d import bitwise_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("szI,szJ,N", [(64, 9, 4), (67, 19, 5), (33, 17, 8), (130, 21, 9),
                                       (19, 13, 21), (19, 13, 63), (19, 13, 64), (19, 13, 65)])
def test_maxflux_omega_levels(szI, szJ, N):
    import torch
    from sailfish_amd import mod_operators as ops
    from sailfish_amd.main3d import initial_depths
    from sailfish_amd.model2d import build_model3d

    print(f"[case] level waves {szI}x{szJ}x{N}", file=sys.stderr, flush=True)
    cfg = configs.random_smooth(szI, szJ, seed=szI + N)
    _ct, GRID, OCEAN, BOUNDARY = build_model3d(cfg, N=N, ndtfast=4, dt=8.0, fix_q5=True)
    initial_depths(GRID, OCEAN)
    c = ops.ctx_of(GRID)
    rng = np.random.default_rng(N)
    S2 = szI * szJ
    host = {n: rng.standard_normal((N + 1, S2)) for n in ("u", "v", "Huon", "Hvom", "W")}
    dev = {n: torch.from_numpy(a.ravel()).cuda() for n, a in host.items()}
    get = lambda t: t.detach().cpu().numpy()
    Hz, z_w = get(GRID.Hz).reshape(N, S2), get(GRID.z_w).reshape(N + 1, S2)
    BC = BOUNDARY.device_maps()["bcIdxFieldIdx2"]
    ops.set_maxflux(None, None, (dev["u"], dev["v"], dev["Huon"], dev["Hvom"], GRID.Hz.reshape(-1)), ctx=c)
    ops.omega(None, None, (dev["W"], dev["u"], dev["v"], dev["Huon"], dev["Hvom"], GRID.z_w.reshape(-1), BC), ctx=c)
    torch.cuda.synchronize()

    f = np.arange(S2)
    i, j = f % szI, f // szI
    un, vn = f[(i > 1) & (j > 0)], f[(i > 0) & (j > 1) & (j < szJ - 1)]
    on_u, om_v = GRID.host["on_u"].ravel(), GRID.host["om_v"].ravel()
    for K in range(N):
        host["Huon"][K, un] = (((Hz[K, un] + Hz[K, un - 1]) * 0.5) * host["u"][K, un]) * on_u[un]
        host["Hvom"][K, vn] = (((Hz[K, vn] + Hz[K, vn - szI]) * 0.5) * host["v"][K, vn]) * om_v[vn]
    Hu, Hv = host["Huon"].ravel(), host["Hvom"].ravel()
    w = np.zeros(S2)
    on = get(BC).ravel() < 0
    for K in range(1, N):
        b = K * S2 + f
        w = w - ((Hu[b + 1] - Hu[b]) + (Hv[b + szI] - Hv[b]))
        host["W"][K, on] = w[on]
    h = z_w[N - 1] - z_w[0]
    for K in range(1, N):
        host["W"][K, on] = host["W"][K, on] - (w[on] * (z_w[K, on] - z_w[0, on])) / h[on]
    host["W"][0, on] = host["W"][N, on] = 0.0
    for n in ("Huon", "Hvom", "W"):
        assert bitwise_equal(get(dev[n]), host[n].ravel()), n
