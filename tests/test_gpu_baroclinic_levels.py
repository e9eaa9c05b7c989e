"""The tracer step and the pressure gradient at the edges of their rounds of eight levels, their
blocks of 64 columns and the tracers' ghost writes (grids with a single interior row or
column): FP64, bit for bit against the oracle, one tracer at a time and both in one pass."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests.helpers2d import bitwise_equal
from tests.test_gpu_baroclinic import _cfg

pytestmark = pytest.mark.gpu

SIZES = [(64, 9, 4), (67, 19, 7), (33, 17, 8), (130, 21, 9), (19, 13, 16), (19, 13, 17), (3, 12, 5), (12, 3, 5),
         (19, 13, 70)]


def _state(szI, szJ, N):
    """A model with random tracers, fluxes and thicknesses, and the oracle's view of it."""
    from oracle import oracle as O
    from oracle import oracle3d as O3
    import torch
    from sailfish_amd.baroclinic import Tracers
    from sailfish_amd.main3d import initial_depths
    from sailfish_amd.model2d import build_model3d
    cfg = _cfg(szI, szJ, N, seed=szI + N)
    _ct, GRID, OCEAN, _B = build_model3d(cfg, N=N, ndtfast=6, dt=12.0)
    initial_depths(GRID, OCEAN)
    S2, rng = szI * szJ, np.random.default_rng(N)
    a = dict(T=10.0 + 5.0 * rng.random(N * S2), S=35.0 + rng.standard_normal(N * S2),
             Hu=40.0 * rng.standard_normal((N + 1) * S2), Hv=40.0 * rng.standard_normal((N + 1) * S2))
    tr = Tracers(GRID, OCEAN, T=a["T"].reshape(N, szJ, szI), S=a["S"].reshape(N, szJ, szI), Scoef=7.6e-4)
    OCEAN.Huon.copy_(torch.from_numpy(a["Hu"].reshape(OCEAN.Huon.shape)))
    OCEAN.Hvom.copy_(torch.from_numpy(a["Hv"].reshape(OCEAN.Hvom.shape)))
    host = GRID.host
    g = O.OGrid(szI, szJ, N, dict(h=cfg["h"], pm=cfg["pm"], pn=cfg["pn"], on_u=host["on_u"], om_v=host["om_v"]))
    BC = -np.ones(S2, np.int32)
    m = O3.OModel3(g, N, host["fomn"], host["sc_r"], host["sc_w"], host["Cs_r"], host["Cs_w"], GRID.hc, 2, BC, BC, BC)
    return GRID, OCEAN, tr, m, a, rng


@pytest.mark.parametrize("szI,szJ,N", SIZES)
def test_tracer_step_levels(szI, szJ, N):
    import torch
    from oracle import oracle as O
    from sailfish_amd import _lib
    from sailfish_amd import mod_operators as ops

    print(f"[case] tracer levels {szI}x{szJ}x{N}", file=sys.stderr, flush=True)
    GRID, OCEAN, tr, m, a, rng = _state(szI, szJ, N)
    Hz_old = GRID.Hz.detach().cpu().numpy().ravel().copy()
    Hz_new = Hz_old * (1.0 + 1e-3 * rng.standard_normal(Hz_old.size))
    tr.Hz_old.copy_(torch.from_numpy(Hz_old.reshape(tr.Hz_old.shape)))
    GRID.Hz.copy_(torch.from_numpy(Hz_new.reshape(GRID.Hz.shape)))
    one = torch.zeros_like(tr.T)
    _lib.check(tr.lib.sf_step3d_t(ops.ctx_of(GRID).handle, tr.precision, tr.T.data_ptr(), one.data_ptr(),
                                  OCEAN.Huon.data_ptr(), OCEAN.Hvom.data_ptr(), tr.Hz_old.data_ptr(),
                                  GRID.Hz.data_ptr(), 60.0, _lib.stream_handle(None)), "sf_step3d_t")
    tr.step(GRID, OCEAN, 60.0)
    torch.cuda.synchronize()
    Tn, Sn = np.zeros_like(a["T"]), np.zeros_like(a["S"])
    for old, new in ((a["T"], Tn), (a["S"], Sn)):
        O.lib().sfo_step3d_t(m.cp, O.ptr(old), O.ptr(new), O.ptr(a["Hu"]), O.ptr(a["Hv"]), O.ptr(Hz_old),
                             O.ptr(Hz_new), 60.0)
    get = lambda t: t.detach().cpu().numpy().ravel()
    assert bitwise_equal(get(tr.T), Tn) and bitwise_equal(get(tr.S), Sn) and bitwise_equal(get(one), Tn)


@pytest.mark.parametrize("szI,szJ,N", SIZES)
def test_pressure_gradient_levels(szI, szJ, N):
    import torch
    from oracle import oracle as O

    print(f"[case] pressure gradient levels {szI}x{szJ}x{N}", file=sys.stderr, flush=True)
    GRID, OCEAN, tr, m, a, rng = _state(szI, szJ, N)
    S2 = szI * szJ
    get = lambda t: t.detach().cpu().numpy().ravel()
    Hz = get(GRID.Hz)
    m.z_r[:] = get(GRID.z_r)
    m.z_w[:N * S2 + S2] = get(GRID.z_w)
    ru, rv = rng.standard_normal((N + 1) * S2), rng.standard_normal((N + 1) * S2)
    OCEAN.ru_t2.copy_(torch.from_numpy(ru))
    OCEAN.rv_t2.copy_(torch.from_numpy(rv))
    tr.pressure_gradient(GRID, OCEAN)
    torch.cuda.synchronize()
    rho = np.zeros(N * S2)
    O.lib().sfo_rho_eos(m.cp, O.ptr(a["T"]), O.ptr(a["S"]), *tr.eos, O.ptr(rho))
    O.lib().sfo_prsgrd(m.cp, O.ptr(rho), O.ptr(m.z_r), O.ptr(m.z_w), O.ptr(Hz), tr.g, tr.rho0, O.ptr(ru), O.ptr(rv))
    assert bitwise_equal(get(OCEAN.ru_t2), ru) and bitwise_equal(get(OCEAN.rv_t2), rv)
