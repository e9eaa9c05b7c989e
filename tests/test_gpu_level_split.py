"""Kernels that split a column's levels over waves -- set_maxflux, omega, the pressure gradient,
the tracer step -- in both precisions, at the remainders of their batches and rounds and on
both sides of their choice between one and four level waves (one on grids of at least 262144
columns with few levels).  Bit for bit: FP64 against the oracle or NumPy, FP32 against the same
formulas on the FP32 inputs (set_maxflux in FP32, the others in FP64 and rounded once).  And
a level of few costs no more than a level of many."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from sailfish_amd import configs
from tests.helpers2d import bitwise_equal
from tests.test_gpu_baroclinic import _cfg

pytestmark = pytest.mark.gpu

SMALL = [(67, 19, 4), (33, 17, 7), (130, 21, 9), (19, 13, 17), (19, 13, 33)]
LARGE = [(513, 513, 4), (515, 512, 5), (640, 410, 8), (640, 410, 9), (513, 512, 16), (513, 512, 17)]


def _fields(szI, szJ, N, dt):
    import torch
    cfg = _cfg(szI, szJ, N, seed=szI + N)
    from sailfish_amd.main3d import initial_depths
    from sailfish_amd.model2d import build_model3d
    _ct, GRID, OCEAN, BOUNDARY = build_model3d(cfg, N=N, ndtfast=4, dt=8.0, fix_q5=True,
                                               dtype=torch.float64 if dt == "f64" else torch.float32)
    initial_depths(GRID, OCEAN)
    return cfg, GRID, OCEAN, BOUNDARY


def _np(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("szI,szJ,N", SMALL + LARGE)
def test_maxflux_omega(szI, szJ, N, dt):
    import torch
    from sailfish_amd import mod_operators as ops
    print(f"[case] level split {szI}x{szJ}x{N} {dt}", file=sys.stderr, flush=True)
    T = np.float64 if dt == "f64" else np.float32
    _cfg_, GRID, OCEAN, BOUNDARY = _fields(szI, szJ, N, dt)
    c = ops.ctx_of(GRID)
    rng = np.random.default_rng(N)
    S2 = szI * szJ
    host = {n: rng.standard_normal((N + 1, S2)).astype(T) for n in ("u", "v", "Huon", "Hvom", "W")}
    dev = {n: torch.from_numpy(a.ravel()).cuda() for n, a in host.items()}
    Hz, z_w = _np(GRID.Hz).reshape(N, S2), _np(GRID.z_w).reshape(N + 1, S2)
    BC = BOUNDARY.device_maps()["bcIdxFieldIdx2"]
    ops.set_maxflux(None, None, (dev["u"], dev["v"], dev["Huon"], dev["Hvom"], GRID.Hz.reshape(-1)), ctx=c)
    ops.omega(None, None, (dev["W"], dev["u"], dev["v"], dev["Huon"], dev["Hvom"], GRID.z_w.reshape(-1), BC), ctx=c)
    torch.cuda.synchronize()
    f = np.arange(S2)
    i, j = f % szI, f // szI
    un, vn = f[(i > 1) & (j > 0)], f[(i > 0) & (j > 1) & (j < szJ - 1)]
    on_u, om_v = GRID.host["on_u"].ravel().astype(T), GRID.host["om_v"].ravel().astype(T)
    for K in range(N):
        host["Huon"][K, un] = (((Hz[K, un] + Hz[K, un - 1]) * T(0.5)) * host["u"][K, un]) * on_u[un]
        host["Hvom"][K, vn] = (((Hz[K, vn] + Hz[K, vn - szI]) * T(0.5)) * host["v"][K, vn]) * om_v[vn]
    Hu, Hv, z = (a.ravel().astype(np.float64) for a in (host["Huon"], host["Hvom"], z_w))
    z = z.reshape(N + 1, S2)
    on = _np(BC).ravel() < 0
    w, sums = np.zeros(S2), []
    for K in range(1, N):
        b = K * S2 + f
        w = w - ((Hu[b + 1] - Hu[b]) + (Hv[b + szI] - Hv[b]))
        sums.append(w)
    h = z[N - 1] - z[0]
    for K in range(1, N):
        host["W"][K, on] = (sums[K - 1][on] - (w[on] * (z[K, on] - z[0, on])) / h[on]).astype(T)
    host["W"][0, on] = host["W"][N, on] = 0.0
    for n in ("Huon", "Hvom", "W"):
        assert bitwise_equal(_np(dev[n]), host[n].ravel()), n


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("szI,szJ,N", SMALL + LARGE)
def test_tracers_and_pressure_gradient(szI, szJ, N, dt):
    import torch
    from oracle import oracle as O
    from oracle import oracle3d as O3
    from sailfish_amd.baroclinic import Tracers
    print(f"[case] level split tracers {szI}x{szJ}x{N} {dt}", file=sys.stderr, flush=True)
    T = np.float64 if dt == "f64" else np.float32
    cfg, GRID, OCEAN, _B = _fields(szI, szJ, N, dt)
    S2, rng = szI * szJ, np.random.default_rng(N)
    r = lambda n, scale, shift=0.0: (shift + scale * rng.standard_normal(n * S2)).astype(T)
    a = dict(T=r(N, 2.0, 10.0), S=r(N, 1.0, 35.0), Hu=r(N + 1, 40.0), Hv=r(N + 1, 40.0), ru=r(N + 1, 1.0), rv=r(N + 1, 1.0))
    tr = Tracers(GRID, OCEAN, T=a["T"].reshape(N, szJ, szI), S=a["S"].reshape(N, szJ, szI), Scoef=7.6e-4)
    put = lambda t, x: t.copy_(torch.from_numpy(x.reshape(t.shape)))
    put(OCEAN.Huon, a["Hu"]), put(OCEAN.Hvom, a["Hv"]), put(OCEAN.ru_t2, a["ru"]), put(OCEAN.rv_t2, a["rv"])
    host = GRID.host
    g = O.OGrid(szI, szJ, N, dict(h=cfg["h"], pm=cfg["pm"], pn=cfg["pn"], on_u=host["on_u"], om_v=host["om_v"]))
    BC = -np.ones(S2, np.int32)
    m = O3.OModel3(g, N, host["fomn"], host["sc_r"], host["sc_w"], host["Cs_r"], host["Cs_w"], GRID.hc, 2, BC, BC, BC)
    d = {k: x.astype(np.float64) for k, x in a.items()}
    wide = lambda t: _np(t).ravel().astype(np.float64)
    Hz = wide(GRID.Hz)
    m.z_r[:], m.z_w[:(N + 1) * S2] = wide(GRID.z_r), wide(GRID.z_w)

    tr.pressure_gradient(GRID, OCEAN)
    torch.cuda.synchronize()
    rho = np.zeros(N * S2)
    O.lib().sfo_rho_eos(m.cp, O.ptr(d["T"]), O.ptr(d["S"]), *tr.eos, O.ptr(rho))
    rho = rho.astype(T).astype(np.float64)
    O.lib().sfo_prsgrd(m.cp, O.ptr(rho), O.ptr(m.z_r), O.ptr(m.z_w), O.ptr(Hz), tr.g, tr.rho0, O.ptr(d["ru"]),
                       O.ptr(d["rv"]))
    for n in ("ru", "rv"):
        assert bitwise_equal(_np(getattr(OCEAN, f"{n}_t2")).ravel(), d[n].astype(T)), n

    Hz_new = (Hz * (1.0 + 1e-3 * rng.standard_normal(Hz.size))).astype(T)
    put(tr.Hz_old, Hz.astype(T)), put(GRID.Hz, Hz_new)
    tr.step(GRID, OCEAN, 60.0)
    torch.cuda.synchronize()
    Hn = Hz_new.astype(np.float64)
    for n in ("T", "S"):
        new = np.zeros_like(d[n])
        O.lib().sfo_step3d_t(m.cp, O.ptr(d[n]), O.ptr(new), O.ptr(d["Hu"]), O.ptr(d["Hv"]), O.ptr(Hz), O.ptr(Hn), 60.0)
        assert bitwise_equal(_np(getattr(tr, n)).ravel(), new.astype(T)), n


@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_few_levels_on_a_large_grid(dt):
    """3000 x 1500: a level of a 4-level grid costs what a level of a 12-level grid does (0.9 to
    1.2 times measured); with four waves on every column it cost up to 1.8 times that."""
    import torch
    from sailfish_amd import mod_operators as ops
    from sailfish_amd.baroclinic import Tracers
    print(f"[case] few levels, large grid {dt}", file=sys.stderr, flush=True)

    def us(fn):
        t = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                fn()
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b) * 100.0)
        return sorted(t)[3]

    level = {}
    for N in (4, 12):
        _c, GRID, OCEAN, BOUNDARY = _fields(3000, 1500, N, dt)
        tr = Tracers(GRID, OCEAN)
        c, BC = ops.ctx_of(GRID), BOUNDARY.device_maps()["bcIdxFieldIdx2"]
        Hu, Hv, W = OCEAN.Huon.reshape(-1), OCEAN.Hvom.reshape(-1), OCEAN.W.reshape(-1)
        Hz, z_w = GRID.Hz.reshape(-1), GRID.z_w.reshape(-1)
        level[N] = [t / N for t in (
            us(lambda: ops.set_maxflux(None, None, (OCEAN.u_t2, OCEAN.v_t2, Hu, Hv, Hz), ctx=c)),
            us(lambda: ops.omega(None, None, (W, OCEAN.u_t2, OCEAN.v_t2, Hu, Hv, z_w, BC), ctx=c)),
            us(lambda: tr.pressure_gradient(GRID, OCEAN)))]
    ratio = [a / b for a, b in zip(level[4], level[12])]
    print(f"[few levels] {dt} set_maxflux, omega, prsgrd: {ratio}", file=sys.stderr, flush=True)
    assert max(ratio) < 1.45, ratio


def test_deep_omega_reads_its_own_chiplets_fluxes():
    """24 x 18 x 100, deeper than the split form of omega takes: set_maxflux and omega after each
    other against each alone, repeated.  Columns on the same XCD in both read the fluxes from
    that XCD's L2: 1.3 times; on different ones it took 1.9."""
    import torch
    from sailfish_amd import mod_operators as ops
    print("[case] deep omega after set_maxflux", file=sys.stderr, flush=True)
    _c, GRID, OCEAN, BOUNDARY = _fields(24, 18, 100, "f64")
    c, BC = ops.ctx_of(GRID), BOUNDARY.device_maps()["bcIdxFieldIdx2"]
    Hu, Hv, W = OCEAN.Huon.reshape(-1), OCEAN.Hvom.reshape(-1), OCEAN.W.reshape(-1)
    Hz, z_w = GRID.Hz.reshape(-1), GRID.z_w.reshape(-1)
    maxflux = lambda: ops.set_maxflux(None, None, (OCEAN.u_t2, OCEAN.v_t2, Hu, Hv, Hz), ctx=c)
    omega = lambda: ops.omega(None, None, (W, OCEAN.u_t2, OCEAN.v_t2, Hu, Hv, z_w, BC), ctx=c)

    def us(*fns):
        g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for fn in fns:
                fn()
            with torch.cuda.graph(g, stream=s):
                for _ in range(20):
                    for fn in fns:
                        fn()
        t = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            g.replay()
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b) * 50.0)
        return sorted(t)[3]

    ratio = us(maxflux, omega) / (us(maxflux) + us(omega))
    print(f"[deep omega] {ratio}", file=sys.stderr, flush=True)
    assert ratio < 1.6, ratio
