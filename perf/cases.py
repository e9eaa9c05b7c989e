"""The work a user of this framework has it do, as cases that can be timed.

Families (``kind``) and what each stands for:

  barotropic  physics-mode 2D run (``phys2d.run_phys``): the barotropic mode of a basin,
              from the 128 x 64 test basin, where a substep is a few microseconds, to
              basins far beyond the last-level cache; FP64 and FP32 state
  reference   the reference's own step2d discretisation (``main2d``, fused substep), FP64
  open        a regional basin with four open edges and the volume constraint
  ensemble    many basins of uneven sizes advanced together (captured substeps, replayed)
  train       Adam steps of the learned closure on mini-batches
  closure     coarse run with the closure network inside the substep
  rhs3d       set_maxflux, omega and rhs3d of one baroclinic step
  main3d      one whole baroclinic step of the reference's loop, FP64
  coupled     one whole coupled baroclinic step with pressure gradient and tracers

``exact`` restates every family in plain torch, in 64 bits.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch

G = 10.0            # gravity of the scheme, m/s2
RHO0 = 1025.0
RDRG = 3e-4
NIN, IN, HID, NOUT = 45, 48, 64, 2
EOS = (1027.0, 14.0, 35.0, 1.7e-4, 7.6e-4)     # R0, T0, S0, Tcoef, Scoef
DT = {"f32": torch.float32, "f64": torch.float64}


def listed() -> list:
    return [
        # the smallest run in use: a 128 x 64 basin over one averaging interval
        dict(name="barotropic_128x64_f64", kind="barotropic", szI=128, szJ=64, dtype="f64", nsub=30),
        # a mid-size basin with odd extents, single precision
        dict(name="barotropic_513x255_f32", kind="barotropic", szI=513, szJ=255, dtype="f32", nsub=30),
        # the benchmark basin
        dict(name="barotropic_2048x1024_f32", kind="barotropic", szI=2048, szJ=1024, dtype="f32", nsub=12),
        # a basin beyond the last-level cache in the reference's precision
        dict(name="barotropic_4096x4096_f64", kind="barotropic", szI=4096, szJ=4096, dtype="f64", nsub=3),
        # the reference's discretisation on a basin of ordinary, odd size
        dict(name="reference_1023x511_f64", kind="reference", szI=1023, szJ=511, dtype="f64", nsub=12),
        # a regional run: all edges open, volume conserved
        dict(name="open_512x256_f64", kind="open", szI=512, szJ=256, dtype="f64", nsub=12),
        # an uneven ensemble
        dict(name="ensemble_21_f32", kind="ensemble", members=21, dtype="f32", nsub=12),
        # closure training: mini-batches at the size the training run uses
        dict(name="train_131072", kind="train", batch=131072, steps=4),
        # the coarse model that the closure serves
        dict(name="closure_512x256_f32", kind="closure", szI=512, szJ=256, dtype="f32", nsub=30),
        # the 3D right-hand side at the 3D workload's size
        dict(name="rhs3d_1024x512x32_f64", kind="rhs3d", szI=1024, szJ=512, N=32, dtype="f64"),
        # the reference's baroclinic loop on a deep column count (over 32 levels)
        dict(name="main3d_386x258x40_f64", kind="main3d", szI=386, szJ=258, N=40, dtype="f64", ndtfast=30),
        # the coupled model's step at the 3D workload's size
        dict(name="coupled_1024x512x32_f32", kind="coupled", szI=1024, szJ=512, N=32, dtype="f32", ndtfast=40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, lo, hi):
    """szI, szJ of about lo..hi points, aspect 1:2 to 3:1; any remainder of the tile widths."""
    pts, asp = _log_int(rng, lo, hi), rng.uniform(0.5, 3.0)
    return max(24, int(math.sqrt(pts * asp))), max(18, int(math.sqrt(pts / asp)))


def draw(rng) -> dict:
    kind = rng.choice(["barotropic"] * 4 + ["reference", "open", "ensemble", "train", "closure", "rhs3d", "main3d",
                                            "coupled", "coupled"])
    dtype = rng.choice(["f32", "f64"])
    if kind == "barotropic":
        szI, szJ = _shape(rng, 4_000, 12_000_000)
        return dict(kind=kind, szI=szI, szJ=szJ, dtype=dtype, nsub=rng.randint(3, 30) if szI * szJ < 1_000_000 else 3)
    if kind == "reference":
        szI, szJ = _shape(rng, 4_000, 2_000_000)
        return dict(kind=kind, szI=szI, szJ=szJ, dtype="f64", nsub=rng.randint(3, 20))
    if kind == "open":
        szI, szJ = _shape(rng, 4_000, 1_000_000)
        return dict(kind=kind, szI=szI, szJ=szJ, dtype=dtype, nsub=rng.randint(3, 20))
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(3, 21), dtype=dtype, nsub=3 * rng.randint(1, 4))
    if kind == "train":
        return dict(kind=kind, batch=64 * _log_int(rng, 16, 2048), steps=rng.randint(1, 4))
    if kind == "closure":
        szI, szJ = _shape(rng, 8_000, 600_000)
        return dict(kind=kind, szI=szI, szJ=szJ, dtype=dtype, nsub=rng.randint(3, 30))
    szI, szJ = _shape(rng, 4_000, 300_000)
    N = rng.choice([10, 16, 20, 30, 31, 32, 36, 48])
    if kind == "rhs3d":
        return dict(kind=kind, szI=szI, szJ=szJ, N=N, dtype=dtype)
    return dict(kind=kind, szI=szI, szJ=szJ, N=N, dtype=dtype if kind == "coupled" else "f64",
                ndtfast=rng.choice([12, 20, 30, 40]))


# ----------------------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------------------
def _modes(rng, szJ, szI, n=4, kmax=6):
    """Smooth random field of unit size: n separable waves with random phases."""
    x = np.arange(szI) / szI
    y = np.arange(szJ) / szJ
    out = np.zeros((szJ, szI))
    for _ in range(n):
        kx, ky = rng.uniform(0.5, kmax, size=2)
        px, py = rng.uniform(0, 2 * np.pi, size=2)
        a = rng.uniform(0.5, 1.0)
        out += np.outer(a * np.sin(2 * np.pi * ky * y + py), np.sin(2 * np.pi * kx * x + px))
    return out / math.sqrt(n / 4.0) / 2.0


def _window(szJ, szI):
    """0 on and outside the walls, 1 inside: initial velocities are at rest there."""
    x = np.sin(np.pi * np.clip((np.arange(szI) - 1.0) / (szI - 2.0), 0, 1))
    y = np.sin(np.pi * np.clip((np.arange(szJ) - 1.0) / (szJ - 2.0), 0, 1))
    return np.outer(y, x)


def _basin(szI, szJ, seed, deep: bool, dx: float, dt: float, vel: float = 0.1, bump: float = 0.05):
    """A closed basin: smooth random bathymetry (200..4000 m, or 100..1000 m), slightly
    stretched metrics, beta plane, wind, a smooth free surface and smooth currents."""
    rng = np.random.Generator(np.random.PCG64(seed))
    lo, hi = (200.0, 4000.0) if deep else (100.0, 1000.0)
    mid, amp = 0.5 * (lo + hi), 0.25 * (hi - lo)
    h = np.clip(mid + amp * _modes(rng, szJ, szI), lo, hi)
    pm = 1.0 / (dx * (1.0 + 0.05 * np.tanh(_modes(rng, szJ, szI, n=2, kmax=2))))
    pn = 1.0 / (dx * (1.0 + 0.05 * np.tanh(_modes(rng, szJ, szI, n=2, kmax=2))))
    y = (np.arange(szJ) - 0.5) * dx
    f = np.broadcast_to((1e-4 + 2e-11 * y)[:, None], (szJ, szI)).copy()
    w = _window(szJ, szI)
    tau = rng.uniform(0.05, 0.15)
    sustr = np.broadcast_to((tau * np.cos(2 * np.pi * y / (szJ * dx)) / RHO0)[:, None], (szJ, szI)).copy()
    return dict(name="basin", szI=szI, szJ=szJ, dx=dx, dy=dx, h=h, f=f, pm=pm, pn=pn, sustr=sustr,
                svstr=0.3 * tau / RHO0 * _modes(rng, szJ, szI, n=2, kmax=2),
                zeta0=bump * _modes(rng, szJ, szI), ubar0=vel * w * _modes(rng, szJ, szI),
                vbar0=vel * w * _modes(rng, szJ, szI), dtfast=dt, rdrg=RDRG)


ENSEMBLE_SIZES = ((256, 128), (384, 256), (512, 256), (768, 384), (1024, 512))


def _member_sizes(case):
    rng = np.random.Generator(np.random.PCG64(case["members"]))
    return [ENSEMBLE_SIZES[int(rng.integers(0, 5))] for _ in range(case["members"])]


def _config(case, seed):
    k = case["kind"]
    if k == "barotropic":
        return _basin(case["szI"], case["szJ"], seed, True, 2e3, 5.0)
    if k == "reference":
        # a short step: the reference's scheme grows slowly (its momentum corrector is void)
        return _basin(case["szI"], case["szJ"], seed, True, 2e3, 0.25, vel=0.0)
    if k == "open":
        return _basin(case["szI"], case["szJ"], seed, True, 2e3, 5.0)
    if k == "closure":
        return _basin(case["szI"], case["szJ"], seed, False, 1250.0, 5.0)
    if k == "ensemble":
        return [_basin(a, b, 1000 * seed + m + 1, False, 5e3, 20.0) for m, (a, b) in enumerate(_member_sizes(case))]
    # 3D: the shallow recipe with currents in the 3D velocity (rhs3d, main3d) or at rest (coupled)
    if k in ("rhs3d", "main3d"):
        c = _basin(case["szI"], case["szJ"], seed, False, 5e3, 7.5 if k == "rhs3d" else 0.25, vel=0.05)
        shear = (0.5 + np.arange(case["N"] + 1) / case["N"])[:, None, None]
        c["u0"], c["v0"] = (shear * c.pop(n)[None] for n in ("ubar0", "vbar0"))
        return c
    c = _basin(case["szI"], case["szJ"], seed, False, 5e3, 7.5, vel=0.0)
    c["h"] = 550.0 + 0.4 * (c["h"] - 550.0)       # gentle slopes for the pressure gradient
    return c


def _open_ext(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed + 77))
    n = (case["szJ"], case["szJ"], case["szI"], case["szI"])
    wave = lambda m: np.sin(2 * np.pi * (np.arange(m) / m * rng.uniform(1, 4) + rng.uniform()))
    return [0.02 * wave(m) for m in n], [0.03 * wave(m) for m in n]


def _stretch(N, theta_s=5.0, theta_b=0.4):
    """s-levels and stretching (Shchepetkin's fourth form), interfaces and midpoints."""
    def Cs(s):
        if s == 0.0:
            return 0.0
        c = (1.0 - math.cosh(theta_s * s)) / (math.cosh(theta_s) - 1.0)
        return (math.exp(theta_b * c) - 1.0) / (1.0 - math.exp(-theta_b))
    sw = [(k - N) / N for k in range(N + 1)]
    sr = [(k + 0.5 - N) / N for k in range(N)]
    Cw = [Cs(s) for s in sw]
    Cw[0], Cw[N] = -1.0, 0.0
    return sr, sw, [Cs(s) for s in sr], Cw


def _tracers(case, seed, cfg):
    """Stratified T and S with a small smooth anomaly, host FP64."""
    rng = np.random.Generator(np.random.PCG64(seed + 5))
    h, hc, N = cfg["h"], 50.0, case["N"]
    sr, _sw, Cr, _Cw = _stretch(N)
    an = _modes(rng, *h.shape)
    T = np.empty((N,) + h.shape)
    S = np.empty_like(T)
    for k in range(N):
        z = h * (hc * sr[k] + Cr[k] * h) / (hc + h)
        e = np.exp(z / 500.0)
        T[k] = 4.0 + 16.0 * e + 0.2 * e * an
        S[k] = 35.0 - 0.3 * e
    return T, S


def _train_data(case, seed):
    """Normalised inputs as BF16 values [n, 48] (columns 45.. zero), targets, mini-batches."""
    g = torch.Generator().manual_seed(seed)
    n = 2 * case["batch"]
    X = torch.zeros((n, IN))
    X[:, :NIN] = torch.randn((n, NIN), generator=g)
    Xb = X.to(torch.bfloat16)
    A = torch.randn((NIN, NOUT), generator=g) / math.sqrt(NIN)
    Y = torch.tanh(X[:, :NIN] @ A) + 0.5 * torch.randn((n, NOUT), generator=g)
    idx = torch.stack([torch.randperm(n, generator=g)[:case["batch"]] for _ in range(case["steps"])]).to(torch.int32)
    return Xb, Y, idx


def _net_params(seed):
    rng = np.random.Generator(np.random.PCG64(seed + 9))
    W1 = np.zeros((IN, HID))
    W1[:NIN] = rng.standard_normal((NIN, HID)) * math.sqrt(2.0 / NIN)
    W2 = rng.standard_normal((HID, HID)) * math.sqrt(2.0 / HID)
    W3 = np.zeros((HID, 16))
    W3[:, :NOUT] = rng.standard_normal((HID, NOUT)) * math.sqrt(1.0 / HID)
    b = 0.1 * rng.standard_normal(2 * HID)
    p = np.concatenate([W1.ravel(), b[:HID], W2.ravel(), b[HID:], W3.ravel(), np.zeros(16)])
    return p.astype(np.float32)


YNORM = (0.0, 2.7e-8, 0.0, 1.2e-8)      # spread of the subgrid tendencies, m/s2


def _norm(case, cfg):
    """Per-feature mean and spread of the initial state (FP32 values)."""
    F = _features(*(torch.from_numpy(np.ascontiguousarray(cfg[k])) for k in ("ubar0", "vbar0", "zeta0", "h", "f")))
    F = F[:, 1:-1, 1:-1].reshape(NIN, -1)
    mu, sd = F.mean(1), F.std(1)
    sd = torch.where(sd > 1e-5 * F.abs().mean(1) + 1e-30, sd, torch.ones_like(sd))
    return mu.float().numpy(), sd.float().numpy()


# ----------------------------------------------------------------------------------------
# what a program holds before the call, and the call
# ----------------------------------------------------------------------------------------
def prepare(case, seed):
    k = case["kind"]
    s = SimpleNamespace(case=case)
    if k == "train":
        from sailfish_amd import closure as CL
        Xb, Y, idx = _train_data(case, seed)
        s.net = CL.ClosureMLP(max_blocks=max(case["batch"] // 64, 1), params=_net_params(seed))
        s.X, s.Y, s.idx = CL.to_bf16_bits(Xb.float()).cuda(), Y.cuda(), [i.contiguous().cuda() for i in idx]
        return s
    cfg = _config(case, seed)
    dt = DT[case["dtype"]]
    if k == "ensemble":
        from sailfish_amd.ensemble import Member, PhysEnsemble
        s.members = [Member(c, dtype=dt) for c in cfg]
        s.ens = PhysEnsemble(s.members, dt)
        s.stream = torch.cuda.Stream()
        s.stream.wait_stream(torch.cuda.current_stream())
        s.ens.capture(s.members[0].ct.weight1[:case["nsub"]].tolist(), s.stream)
        torch.cuda.current_stream().wait_stream(s.stream)
        return s
    if k in ("barotropic", "open"):
        from sailfish_amd.model2d import build_model
        from sailfish_amd.phys2d import PhysStepper
        s.ct, s.grid, s.ocean, s.bry = build_model(cfg, dtype=dt, ndtfast=30)
        if k == "open":
            ez, eu = _open_ext(case, seed)
            s.st = PhysStepper(s.grid, s.ocean, rdrg=RDRG, open_edges=15, volcons=True, zeta_ext=ez, vel_ext=eu)
        else:
            s.st = PhysStepper(s.grid, s.ocean, rdrg=RDRG)
        return s
    if k == "reference":
        from sailfish_amd.model2d import build_model
        s.ct, s.grid, s.ocean, s.bry = build_model(cfg, dtype=dt, ndtfast=30, fix_q5=True)
        return s
    if k == "closure":
        from sailfish_amd import closure as CL
        s.model = CL.Model(cfg, dtype=dt)
        s.model.n = 1                              # a run under way, not its Euler start
        s.net = CL.ClosureMLP(params=_net_params(seed))
        s.net.set_norm(*_norm(case, cfg), np.array(YNORM, np.float32))
        return s
    from sailfish_amd.model2d import build_model3d
    nd = case.get("ndtfast", 30)
    s.ct, s.grid, s.ocean, s.bry = build_model3d(cfg, N=case["N"], ndtfast=nd, dt=nd * cfg["dtfast"], dtype=dt)
    s.bry.device_maps()
    if k == "coupled":
        from sailfish_amd.coupled3d import main3d_coupled
        T, S = _tracers(case, seed, cfg)
        R0, T0, S0, Tc, Sc = EOS
        s.cs = main3d_coupled(s.ct, s.grid, s.ocean, s.bry, 0, rdrg=RDRG,
                              tracers=dict(T=T, S=S, R0_=R0, T0_=T0, S0_=S0, Tcoef=Tc, Scoef=Sc))
        return s
    from sailfish_amd import mod_operators as ops
    from sailfish_amd.main3d import Main3dState, initial_depths
    s.m3 = Main3dState(s.grid, s.ocean)
    ops.setVerticalVelEq(None, None, (s.m3.eqSD, s.m3.eqD, s.m3.eqRHS), ctx=ops.ctx_of(s.grid))
    initial_depths(s.grid, s.ocean)
    return s


def _state2d(o):
    return {n: getattr(o, n) for n in ("zeta", "ubar", "vbar", "rzeta", "rubar", "rvbar", "Zt_avg1", "DU_avg1",
                                       "DV_avg1")}


def run(s):
    case, k = s.case, s.case["kind"]
    if k in ("barotropic", "open"):
        from sailfish_amd.phys2d import run_phys
        s.ct.first2DTimeStep()
        run_phys(s.ct, s.grid, s.ocean, case["nsub"], s.st, start_first=False)
        return _state2d(s.ocean)
    if k == "reference":
        from sailfish_amd.main2d import main2d
        s.ct.first2DTimeStep()
        main2d(s.ct, s.grid, s.ocean, s.bry, case["nsub"], fused=True)
        o = s.ocean
        return dict(zeta=o.zeta, ubar=o.ubar_t2, vbar=o.vbar_t2, Zt_avg1=o.Zt_avg1, DU_avg1=o.DU_avg1,
                    DV_avg1=o.DV_avg1)
    if k == "ensemble":
        s.ens.replay()
        s.ens.sync()
        return [(m.OCEAN.zeta, m.OCEAN.ubar, m.OCEAN.vbar) for m in s.members]
    if k == "train":
        for i in s.idx:
            s.net.train_step(s.X, s.Y, i, lr=1e-3)
        return s.net.get_params()
    if k == "closure":
        s.model.ct.first2DTimeStep()
        for _ in range(case["nsub"]):
            s.model.step(s.net)
        return _state2d(s.model.OCEAN)
    o, g = s.ocean, s.grid
    if k == "rhs3d":
        from sailfish_amd import mod_operators as ops
        from sailfish_amd.rhs import rhs3d
        c, BC = ops.ctx_of(g), s.bry.device_maps()["bcIdxFieldIdx2"]
        Hu, Hv, W = o.Huon.reshape(-1), o.Hvom.reshape(-1), o.W.reshape(-1)
        ops.set_maxflux(None, None, (o.u_t2, o.v_t2, Hu, Hv, g.Hz.reshape(-1)), ctx=c)
        ops.omega(None, None, (W, o.u_t2, o.v_t2, Hu, Hv, g.z_w.reshape(-1), BC), ctx=c)
        rhs3d(g, o, s.bry)
        return dict(Huon=Hu, Hvom=Hv, W=W, ru=o.ru_t2, rv=o.rv_t2)
    out3 = dict(u=o.u_t2, v=o.v_t2, ru=o.ru_t2, rv=o.rv_t2, Huon=o.Huon, Hvom=o.Hvom, W=o.W, Hz=g.Hz, z_w=g.z_w,
                z_r=g.z_r, Zt_avg1=o.Zt_avg1, DU_avg1=o.DU_avg1, DV_avg1=o.DV_avg1, zeta=o.zeta)
    if k == "main3d":
        from sailfish_amd.main3d import baroclinic_step
        baroclinic_step(s.ct, g, o, s.bry, s.m3, fused=True)
        return dict(out3, ubar=o.ubar_t2, vbar=o.vbar_t2)
    from sailfish_amd.coupled3d import coupled_step
    coupled_step(s.ct, g, o, s.bry, s.cs)
    t = s.cs.tracers
    return dict(out3, ubar=o.ubar, vbar=o.vbar, T=t.T, S=t.S, rho=t.rho, DU_avg2=s.cs.DU_avg2, DV_avg2=s.cs.DV_avg2)


# ----------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------
def work(case) -> dict:
    """Bytes of the fields a substep (or a 3D kernel chain) reads and writes once, and
    its arithmetic.  A substep reads six static fields, two time levels of three fields and
    one of three right-hand sides, writes one level of each, and updates three FP64 sums."""
    k = case["kind"]
    e = 8 if case.get("dtype") == "f64" else 4
    sub = 21 * e + 48                        # bytes a point, physics substep
    flop = 330
    if k == "train":
        n = case["batch"] * case["steps"]
        return dict(bytes=n * (2 * IN + 4 * NOUT + 4), flops=n * 6 * (IN * HID + HID * HID + HID * NOUT))
    if k == "ensemble":
        pts = sum(a * b for a, b in _member_sizes(case))
        return dict(bytes=pts * sub * case["nsub"], flops=pts * flop * case["nsub"])
    S2 = case["szI"] * case["szJ"]
    if k in ("barotropic", "open"):
        return dict(bytes=S2 * sub * case["nsub"], flops=S2 * flop * case["nsub"])
    if k == "closure":
        net = 2 * (NIN * HID + HID * HID + HID * NOUT)
        return dict(bytes=S2 * (sub + e) * case["nsub"], flops=S2 * (flop + net) * case["nsub"])
    if k == "reference":
        return dict(bytes=S2 * (16 * e + 48) * case["nsub"], flops=S2 * 90 * case["nsub"])
    n3 = S2 * case["N"]
    if k == "rhs3d":
        # in: u, v, Hz, z_w; out: Huon, Hvom, W, ru, rv
        return dict(bytes=n3 * 9 * e, flops=n3 * 200)
    nsub = int(1.45 * case["ndtfast"])
    if k == "main3d":
        # in: u, v, AKv, Hz, z_w; out: u, v, ru, rv, Huon, Hvom, W, Hz, z_w, z_r
        return dict(bytes=n3 * 15 * e + S2 * (16 * e + 48) * nsub, flops=n3 * 300 + S2 * 90 * nsub)
    # as main3d, with T, S in and out, rho out, and two older right-hand sides of u and v in
    return dict(bytes=n3 * 25 * e + S2 * (sub + 64) * nsub, flops=n3 * 450 + S2 * flop * nsub)


# ----------------------------------------------------------------------------------------
# 64-bit restatement
# ----------------------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _sh(a, o):
    """b[f] = a[f + o] on a flat array, zero outside."""
    if o == 0:
        return a
    b = torch.zeros_like(a)
    if o > 0:
        b[:-o] = a[o:]
    else:
        b[-o:] = a[:o]
    return b


def _sh2(a, dj, di):
    b = torch.zeros_like(a)
    J, I = a.shape
    b[max(0, -dj):J - max(0, dj), max(0, -di):I - max(0, di)] = \
        a[max(0, dj):J - max(0, -dj), max(0, di):I - max(0, -di)]
    return b


def _features(u, v, z, h, f):
    """[45, J, I]: per field the value and the eight differences neighbour - centre."""
    out = []
    for a in (u, v, z, h, f):
        for dj in (-1, 0, 1):
            for di in (-1, 0, 1):
                out.append(a if dj == 0 and di == 0 else _sh2(a, dj, di) - a)
    return torch.stack(out)


def _weights(ndtfast):
    """The averaging weights of a barotropic interval: the power-law filter with its
    centroid shifted to ndtfast, and the weights of the filtered transport."""
    Fa, Fb, Fg = 2.0, 4.0, 0.284
    w1, w2 = [0.0] * 258, [0.0] * 258
    scale = (Fa + 1.0) * (Fa + Fb + 1.0) / ((Fa + 2.0) * (Fa + Fb + 2.0) * ndtfast)
    gam = Fg * max(0.0, 1.0 - 10.0 / ndtfast)
    nfast = 0
    for _ in range(16):
        nfast = 0
        for i in range(2 * ndtfast):
            x = scale * (i + 1)
            w1[i] = x ** Fa - x ** (Fa + Fb) - gam * x
            if w1[i] > 0.0:
                nfast = i + 1
            if nfast > 0 and w1[i] < 0.0:
                w1[i] = 0.0
        s = sum(w1[:nfast])
        m = sum((i + 1) * w1[i] for i in range(nfast))
        scale = scale * m / (s * ndtfast)
    for _ in range(ndtfast):
        c = ndtfast - sum((i + 1) * w1[i] for i in range(nfast)) / sum(w1[:nfast])
        if c > 1.0:
            nfast += 1
            for i in range(nfast - 1, 1, -1):
                w1[i] = w1[i - 1]
            w1[0] = 0.0
        elif c > 0.0:
            for i in range(nfast - 1, 1, -1):
                w1[i] = (1.0 - c) * w1[i] + c * w1[i - 1]
            w1[0] = (1.0 - c) * w1[0]
        elif c < 0.0:
            for i in range(nfast - 1):
                w1[i] = (1.0 + c) * w1[i] - c * w1[i + 1]
            w1[nfast] = (1.0 + c) * w1[nfast]
    for j in range(nfast):
        for i in range(j):
            w2[i] += w1[j]
    a, b = 1.0 / sum(w1[:nfast]), 1.0 / sum(w2[:nfast])
    for i in range(nfast):
        w1[i] *= a
        w2[i] *= b
    return w1[:257], w2[:257], nfast


class _Basin2D:
    """Static fields (the values the state's precision holds) and the physics substep."""

    def __init__(self, cfg, dtype, open_ext=None, net=None):
        d = _dev()
        self.q = lambda a: torch.from_numpy(np.array(a, dtype=np.float64)).to(d, dtype).double().reshape(-1)
        self.I, self.J = cfg["szI"], cfg["szJ"]
        W, S2 = self.I, self.I * self.J
        q = self.q
        self.h, self.pm, self.pn, self.f = q(cfg["h"]), q(cfg["pm"]), q(cfg["pn"]), q(cfg["f"])
        self.fomn = q(cfg["f"] / (cfg["pm"] * cfg["pn"]))
        self.su, self.sv = q(cfg["sustr"]), q(cfg["svstr"])
        inv = lambda a, o: 2.0 / (_sh(a, o) + a)
        self.onu, self.omu = inv(self.pn, -1), inv(self.pm, -1)
        self.omv, self.onv = inv(self.pm, -W), inv(self.pn, -W)
        n = torch.arange(S2, device=d)
        i, j = n % W, n // W
        L, M = self.I - 1, self.J - 1
        inn = (i >= 1) & (i <= L - 1) & (j >= 1) & (j <= M - 1)
        self.mr, self.mu, self.mv = inn, inn & (i >= 2), inn & (j >= 2)
        self.ext = open_ext
        if open_ext:
            self.ext = [[torch.from_numpy(a).to(d) for a in x] for x in open_ext]
        self.net = net
        z = lambda: [torch.zeros(S2, dtype=torch.float64, device=d) for _ in range(3)]
        ini = lambda k: [q(cfg[k]).clone() for _ in range(3)]
        self.s = dict(zeta=ini("zeta0"), ubar=ini("ubar0"), vbar=ini("vbar0"), rzeta=z(), rubar=z(), rvbar=z())
        self.slot = [0, 1, 2]
        self.Zt, self.DU, self.DV = z()
        self.dt = cfg["dtfast"]

    def rotate(self):
        a, b, c = self.slot
        self.slot = [b, c, a]

    def lev(self, name, k):
        return self.s[name][self.slot[k]]

    def put(self, name, k, value, mask=None):
        a = self.s[name][self.slot[k]]
        self.s[name][self.slot[k]] = value if mask is None else torch.where(mask, value, a)

    def flux(self, z, u, v):
        D = self.h + z
        return (0.5 * (_sh(D, -1) + D)) * u * self.onu, (0.5 * (_sh(D, -self.I) + D)) * v * self.omv

    def rhs_zeta(self, DU, DV):
        return (DU - _sh(DU, 1)) + (DV - _sh(DV, self.I))

    def rhs_u(self, z, u, v, gz, DU, DV, su):
        W, D = self.I, self.h + z
        g0, h0 = _sh(gz, -1), _sh(self.h, -1)
        r = 0.5 * G * self.onu * ((h0 + self.h) * (g0 - gz) + (g0 * g0 - gz * gz))
        fx = 0.25 * (DU + _sh(DU, 1)) * (u + _sh(u, 1))                     # at rho
        fe = 0.25 * (DV + _sh(DV, -1)) * (u + _sh(u, -W))                   # at psi
        r = r - ((fx - _sh(fx, -1)) + (_sh(fe, W) - fe))
        c = 0.5 * D * self.fomn * (v + _sh(v, W))
        return r + 0.5 * (c + _sh(c, -1)) - RDRG * u * self.omu * self.onu + su * self.omu * self.onu

    def rhs_v(self, z, u, v, gz, DU, DV, sv):
        W, D = self.I, self.h + z
        g0, h0 = _sh(gz, -W), _sh(self.h, -W)
        r = 0.5 * G * self.omv * ((h0 + self.h) * (g0 - gz) + (g0 * g0 - gz * gz))
        fx = 0.25 * (DU + _sh(DU, -W)) * (v + _sh(v, -1))                   # at psi
        fe = 0.25 * (DV + _sh(DV, W)) * (v + _sh(v, W))                     # at rho
        r = r - ((_sh(fx, 1) - fx) + (fe - _sh(fe, -W)))
        c = 0.5 * D * self.fomn * (u + _sh(u, 1))
        return r - 0.5 * (c + _sh(c, -W)) - RDRG * v * self.omv * self.onv + sv * self.omv * self.onv

    def bc_z(self, z):
        z = z.view(self.J, self.I)
        z[1:-1, 0], z[1:-1, -1] = z[1:-1, 1], z[1:-1, -2]
        z[0], z[-1] = z[1], z[-2]

    def bc_uv(self, u, v):
        u, v = u.view(self.J, self.I), v.view(self.J, self.I)
        u[:, 0], u[:, 1], u[:, -1] = 0.0, 0.0, 0.0
        u[0, 2:-1], u[-1, 2:-1] = u[1, 2:-1], u[-2, 2:-1]
        v[0], v[1], v[-1] = 0.0, 0.0, 0.0
        v[2:-1, 0], v[2:-1, -1] = v[2:-1, 1], v[2:-1, -2]

    # open edges: (ghost point, interior point, face) per edge west, east, south, north
    def edges(self):
        r = torch.arange(1, self.J - 1, device=self.h.device) * self.I
        c = torch.arange(1, self.I - 1, device=self.h.device)
        L, top = self.I - 1, (self.J - 1) * self.I
        return ((r, r + 1, r + 1), (r + L, r + L - 1, r + L), (c, c + self.I, c + self.I),
                (c + top, c + top - self.I, c + top))

    def open_z(self, zn, zb, dts):
        for e, (g, n, _f) in enumerate(self.edges()):
            m = self.pm if e < 2 else self.pn
            Ce = dts * 0.5 * (m[g] + m[n]) * torch.sqrt(G * (self.h[g] + zb[g]))
            zn[g] = (zb[g] + Ce * zn[n]) / (1.0 + Ce)

    def open_uv(self, zn, u, v):
        I, L, M = self.I, self.I - 1, self.J - 1
        for e, (g, n, f) in enumerate(self.edges()):
            x, sg = (u if e < 2 else v), (-1.0 if e in (0, 2) else 1.0)
            D = 0.5 * ((self.h[g] + zn[g]) + (self.h[n] + zn[n]))
            b = slice(1, len(g) + 1)
            x[f] = self.ext[1][e][b] + sg * torch.sqrt(G / D) * (0.5 * (zn[g] + zn[n]) - self.ext[0][e][b])
            X = x.view(self.J, I)
            if e == 0:
                X[0, 1], X[M, 1] = X[1, 1].clone(), X[M - 1, 1].clone()
            elif e == 1:
                X[0, L], X[M, L] = X[1, L].clone(), X[M - 1, L].clone()
            elif e == 2:
                X[1, 0], X[1, L] = X[1, 1].clone(), X[1, L - 1].clone()
            else:
                X[M, 0], X[M, L] = X[M, 1].clone(), X[M, L - 1].clone()
        # no net flow through the open edges: one uniform correction
        area, flow = 0.0, 0.0
        for e, (_g, _n, f) in enumerate(self.edges()):
            o, met, x = (1, self.onu, u) if e < 2 else (I, self.omv, v)
            a = 0.5 * ((zn[f - o] + self.h[f - o]) + (zn[f] + self.h[f])) * met[f]
            area = area + a.sum()
            flow = flow + (1.0 if e in (0, 2) else -1.0) * (a * x[f]).sum()
        xs = flow / area
        for e, (_g, _n, f) in enumerate(self.edges()):
            x = u if e < 2 else v
            x[f] = x[f] + (-xs if e in (0, 2) else xs)

    def closure_stress(self, z, u, v):
        sh = (self.J, self.I)
        F = _features(u.view(sh), v.view(sh), z.view(sh), self.h.view(sh), self.f.view(sh)).reshape(NIN, -1)
        W1, b1, W2, b2, W3, b3, mu, sd = self.net
        X = (F - mu[:, None]) / sd[:, None]
        A = torch.relu(W1[:NIN].T @ X + b1[:, None])
        A = torch.relu(W2.T @ A + b2[:, None])
        out = W3.T @ A + b3[:, None]
        D = self.h + z
        R = [(out[c] * YNORM[2 * c + 1] + YNORM[2 * c]) * (0.5 * (_sh(D, -o) + D)) for c, o in ((0, 1), (1, self.I))]
        zero = torch.zeros_like(z)
        return self.su + torch.where(self.mu, R[0], zero), self.sv + torch.where(self.mv, R[1], zero)

    def substep(self, w, first=False, cp=None):
        W, dt, lev = self.I, self.dt, self.lev
        z0, z1, u0, u1, v0, v1 = (lev(n, k) for n in ("zeta", "ubar", "vbar") for k in (0, 1))
        pmn = self.pm * self.pn
        csu, csv = self.closure_stress(z1, u1, v1) if self.net else (self.su, self.sv)
        DU, DV = self.flux(z1, u1, v1)
        rz = self.rhs_zeta(DU, DV)
        self.put("rzeta", 1, rz, self.mr)
        rz1 = lev("rzeta", 1)
        zs = torch.where(self.mr, z1 + pmn * dt * rz if first else z0 + pmn * (2.0 * dt) * rz, z1)
        if cp:
            for n, x in (("DU2", DU), ("DV2", DV)):
                cp[n] = torch.where(self.mr, (0.0 if first else cp[n]) + cp["w2p"] * x, cp[n])
        self.bc_z(zs)
        if self.ext:
            self.open_z(zs, z1 if first else z0, dt if first else 2.0 * dt)
        gz = 0.5 * (z1 + zs) if first else (1.0 - 8.0 / 25.0) * z1 + (4.0 / 25.0) * (z0 + zs)
        zb, ub, vb = (z1, u1, v1) if first else (z0, u0, v0)
        c1 = 0.5 * dt if first else dt
        Db, Ds, D1 = self.h + zb, self.h + zs, self.h + z1
        new = []
        for d, o, b, r, m, key, stress in ((0, 1, ub, "rubar", self.mu, "Fu", self.su),
                                           (1, W, vb, "rvbar", self.mv, "Fv", self.sv)):
            x = (self.rhs_v if d else self.rhs_u)(z1, u1, v1, gz, DU, DV, stress)
            if cp:
                if first:
                    F = cp["rvfrc" if d else "rufrc"] - x
                    cp[key] = torch.where(m, F, cp[key])
                x = x + cp[key]                   # first step of a run: no extrapolation
            self.put(r, 1, x, m)
            cff = (self.pm + _sh(self.pm, -o)) * (self.pn + _sh(self.pn, -o))
            new.append(torch.where(m, (b * (Db + _sh(Db, -o)) + cff * c1 * x) / (Ds + _sh(Ds, -o)), (v1 if d else u1)))
        us, vs = new
        self.bc_uv(us, vs)
        if self.ext:
            self.open_uv(zs, us, vs)
        DU, DV = self.flux(zs, us, vs)
        r = self.rhs_zeta(DU, DV)
        z2 = z1 + pmn * (dt * r if first else dt / 12.0 * (5.0 * r + 8.0 * rz1 - lev("rzeta", 0)))
        z2 = torch.where(self.mr, z2, z1)
        self.Zt = torch.where(self.mr, self.Zt + w * zs, self.Zt)
        self.DU = torch.where(self.mr, self.DU + w * DU, self.DU)
        self.DV = torch.where(self.mr, self.DV + w * DV, self.DV)
        if cp:
            cp["DU2"] = torch.where(self.mr, cp["DU2"] + cp["w2c"] * DU, cp["DU2"])
            cp["DV2"] = torch.where(self.mr, cp["DV2"] + cp["w2c"] * DV, cp["DV2"])
        self.bc_z(z2)
        if self.ext:
            self.open_z(z2, z1, dt)
        gz = 0.6 * z2 + 0.4 * zs
        D2 = self.h + z2
        new = []
        for d, o, b, r, m, key, stress in ((0, 1, u1, "rubar", self.mu, "Fu", csu), (1, W, v1, "rvbar", self.mv, "Fv", csv)):
            x = (self.rhs_v if d else self.rhs_u)(zs, us, vs, gz, DU, DV, stress)
            if cp:
                x = x + cp[key]
            cff = (self.pm + _sh(self.pm, -o)) * (self.pn + _sh(self.pn, -o))
            t = 0.5 * dt * (x if first else (5.0 * x + 8.0 * lev(r, 1) - lev(r, 0)) / 12.0)
            new.append(torch.where(m, (b * (D1 + _sh(D1, -o)) + cff * t) / (D2 + _sh(D2, -o)), b))
        self.bc_uv(*new)
        if self.ext:
            self.open_uv(z2, *new)
        for n, x in (("zeta", z2), ("ubar", new[0]), ("vbar", new[1])):
            self.put(n, 2, x)

    def run(self, nsub, w1):
        for n in range(nsub):
            self.rotate()
            self.substep(w1[min(n, 256)])

    def out(self):
        sh = (3, self.J, self.I)
        o = {n: torch.stack(self.s[n]).reshape(sh) for n in self.s}
        return dict(o, Zt_avg1=self.Zt, DU_avg1=self.DU, DV_avg1=self.DV)


class _Reference2D:
    """The reference's step2d (its metrics average along the other axis)."""

    def __init__(self, cfg):
        d = _dev()
        t = lambda a: torch.from_numpy(np.array(a, dtype=np.float64)).to(d)
        self.I, self.J, self.dt = cfg["szI"], cfg["szJ"], cfg["dtfast"]
        self.h, self.pm, self.pn = t(cfg["h"]).reshape(-1), t(cfg["pm"]).reshape(-1), t(cfg["pn"]).reshape(-1)
        on, om = torch.zeros_like(t(cfg["pn"])), torch.zeros_like(t(cfg["pn"]))
        pm, pn = t(cfg["pm"]), t(cfg["pn"])
        on[1:] = 2.0 / (pn[:-1] + pn[1:])
        om[:, 1:] = 2.0 / (pm[:, :-1] + pm[:, 1:])
        self.onu, self.omv = on.reshape(-1), om.reshape(-1)
        n = torch.arange(self.I * self.J, device=d)
        i, j = n % self.I, n // self.I
        self.inn = (i > 0) & (i < self.I - 1) & (j > 0) & (j < self.J - 1)
        self.rn = (i > 0) & (j > 0)
        z = lambda: [torch.zeros_like(self.h) for _ in range(3)]
        self.z, self.u, self.v = [t(cfg["zeta0"]).reshape(-1).clone() for _ in range(3)], z(), z()
        self.rz = z()
        self.slot = [0, 1, 2]
        self.Zt, self.DU, self.DV = z()

    def rhs_zeta(self, z, u, v, w=None):
        W, D = self.I, self.h + z
        DU, DV = u * (0.5 * (D + _sh(D, -1))), v * (0.5 * (D + _sh(D, -W)))
        fu, fv = DU * self.onu, DV * self.omv
        r = ((_sh(fu, 1) - fu) + (_sh(fv, W) - fv)) * self.pm * self.pn
        if w is not None:
            self.Zt = torch.where(self.inn, self.Zt + w * z, self.Zt)
            self.DU = torch.where(self.inn, self.DU + w * fu, self.DU)
            self.DV = torch.where(self.inn, self.DV + w * fv, self.DV)
        return r

    def zbc(self, z):
        z = z.view(self.J, self.I)
        z[:-1, 0], z[:-1, -1] = z[:-1, 1].clone(), z[:-1, -2].clone()
        z[0, :-1], z[-1, :-1] = z[1, :-1].clone(), z[-2, :-1].clone()

    def substep(self, w, zero_v=False):
        W, dt = self.I, self.dt
        a, b, c = self.slot
        self.slot = [b, c, a]
        t0, t1, t2 = self.slot
        r = self.rhs_zeta(self.z[t1], self.u[t1], self.v[t1])
        self.rz[t1] = torch.where(self.inn, r, self.rz[t1])
        z2 = torch.where(self.rn, self.z[t0] + dt * self.rz[t1], self.z[t2])
        self.zbc(z2)
        gz = 0.6 * z2 + 0.4 * self.z[t0]
        dg = lambda o: (0.5 * (self.h + _sh(self.h, -o))) * (gz - _sh(gz, -o)) + 0.5 * (gz * gz - _sh(gz, -o) ** 2)
        D1, D2 = self.h + self.z[t1], self.h + z2
        zero = torch.zeros_like(gz)
        new = []
        for o, met, x in ((1, self.onu, self.u), (W, self.omv, self.v)):
            rr = torch.where(self.inn, G * met * dg(o), zero)
            y = (x[t1] * (0.5 * (D1 + _sh(D1, -o))) + dt * rr * self.pm * self.pn) / (0.5 * (D2 + _sh(D2, -o)))
            new.append(torch.where(self.rn, y, x[t2]))
        u, v = new[0].view(self.J, W), new[1].view(self.J, W)
        u[:-1, 1], u[:-1, -1], u[1, 1:-1], u[-1, 1:-1] = 0.0, 0.0, 0.0, 0.0
        v[1:-1, 0], v[1:-1, -1], v[0, :-1], v[-1, :-1] = 0.0, 0.0, 0.0, 0.0
        u, v = new
        r = self.rhs_zeta(z2, u, v, w)
        self.rz[t1] = torch.where(self.inn, r, self.rz[t1])
        z2 = z2 + dt / 12.0 * (5.0 * self.rz[t2] + 8.0 * self.rz[t1] - self.rz[t0])
        self.zbc(z2)
        self.z[t2], self.u[t2], self.v[t2] = z2, u, (torch.zeros_like(v) if zero_v else v)


class _Model3D:
    """The 3D kernels on flat (N+1) x S2 arrays."""

    def __init__(self, case, cfg, dtype):
        d = _dev()
        self.I, self.J, self.N = cfg["szI"], cfg["szJ"], case["N"]
        N, S2 = self.N, self.I * self.J
        self.S2 = S2
        t = lambda a: torch.from_numpy(np.array(a, dtype=np.float64)).to(d).reshape(-1)
        self.h, self.pm, self.pn = t(cfg["h"]), t(cfg["pm"]), t(cfg["pn"])
        self.fomn = t(cfg["f"] / (cfg["pm"] * cfg["pn"]))
        ref = _Reference2D(cfg)
        self.onu, self.omv = ref.onu, ref.omv
        self.sr, self.sw, self.Cr, self.Cw = _stretch(N)
        n = torch.arange(S2, device=d)
        self.i, self.j = n % self.I, n // self.I
        i, j, L, M = self.i, self.j, self.I - 1, self.J - 1
        self.unode, self.vnode = (i > 1) & (j > 0), (i > 0) & (j > 1) & (j < M)
        self.edge = ((i == 0) | (i == L) | (j == 0) | (j == M)) & ~((i == L) & (j == M))
        self.inner = (i > 1) & (i < L - 1) & (j > 1) & (j < M - 1)
        self.cu = (i >= 2) & (i <= L - 1) & (j >= 1) & (j <= M - 1)
        self.cv = (i >= 1) & (i <= L - 1) & (j >= 2) & (j <= M - 1)
        z = lambda k=1: torch.zeros((N + k, S2), dtype=torch.float64, device=d)
        q = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(d, dtype).double().reshape(N + 1, S2)
        self.u, self.v = (q(cfg[k]).clone() if k in cfg else z() for k in ("u0", "v0"))
        self.ru, self.rv, self.Hu, self.Hv, self.W = z(), z(), z(), z(), z()
        zw = torch.stack([self.h * ((50.0 * self.sw[k] + self.Cw[k] * self.h) / (50.0 + self.h)) for k in range(N + 1)])
        zw[N] = 0.0
        self.AKv = (2.0e-3 + 8.0e-3 * torch.exp(zw / 150.0)).to(dtype).double()
        self.dt = case.get("ndtfast", 30) * cfg["dtfast"]

    def depths(self, Zt):
        N = self.N
        c = lambda s, C: (50.0 * s + C * self.h) / (50.0 + self.h)
        self.zw = torch.stack([Zt + (Zt + self.h) * c(self.sw[k], self.Cw[k]) for k in range(N)] + [Zt])
        self.zr = torch.stack([Zt + (Zt + self.h) * c(self.sr[k], self.Cr[k]) for k in range(N)])
        self.Hz = self.zw[1:] - self.zw[:-1]

    def s(self, a, o):
        return _sh(a.reshape(-1), o).view(a.shape)

    def maxflux(self):
        N, W = self.N, self.I
        a = 0.5 * (self.Hz + self.s(self.Hz, -1)) * self.u[:N] * self.onu
        b = 0.5 * (self.Hz + self.s(self.Hz, -W)) * self.v[:N] * self.omv
        self.Hu[:N] = torch.where(self.unode, a, self.Hu[:N])
        self.Hv[:N] = torch.where(self.vnode, b, self.Hv[:N])

    def omega(self):
        N = self.N
        d = (self.s(self.Hu, 1) - self.Hu) + (self.s(self.Hv, self.I) - self.Hv)
        w = torch.zeros_like(self.W)
        w[1:N] = -torch.cumsum(d[1:N], 0)
        ws = w[N - 1].clone()
        w[1:N] = w[1:N] - ws * (self.zw[1:N] - self.zw[0]) / (self.zw[N - 1] - self.zw[0])
        self.W = torch.where(self.edge, self.W, w)

    def rhs(self):
        N, W, S2, s = self.N, self.I, self.S2, self.s
        u, v, Hu, Hv = self.u, self.v, self.Hu, self.Hv
        rn = (self.i > 0) & (self.j > 0)
        ru, rv = torch.zeros_like(u), torch.zeros_like(v)
        Hf = torch.zeros_like(u)
        Hf[:N] = self.Hz * self.fomn
        uf, vf = Hf * 0.5 * (v + s(v, W)), Hf * 0.5 * (u + s(u, 1))
        # a column's Coriolis terms stay on its own level: no carry from the level below at f = 0
        cu, cv = 0.5 * (uf + s(uf, -1)), 0.5 * (vf + s(vf, -W))
        ru[:N] = torch.where(rn, cu[:N], ru[:N])
        rv[:N] = torch.where(rn, -cv[:N], rv[:N])
        dxx = lambda a: s(a, -1) - 2.0 * a + s(a, 1)
        dee = lambda a: s(a, -W) - 2.0 * a + s(a, W)
        av = lambda a, o: 0.5 * (a + s(a, o))
        du, de = dxx(u), dee(u)
        uR, HvP = av(u, 1), av(Hv, -W)
        uxxR = torch.where(uR + s(uR, 1) >= 0, du, s(du, 1))
        ueeP = torch.where(HvP + s(HvP, -W) >= 0, de, s(de, -W))
        # flux + (-1/2 curvature) (mass flux - 1/2 its curvature), at rho and psi
        UFx = uR - 0.5 * uxxR * (av(Hu, 1) - 0.5 * av(dxx(Hu), 1))
        UFe = av(u, -1) - 0.5 * ueeP * (HvP - 0.5 * av(dxx(Hv), -W))
        VFx = av(v, -W) - 0.5 * ueeP * (av(Hu, -1) - 0.5 * av(dee(Hu), -1))
        VFe = av(v, W) - 0.5 * uxxR * (av(Hv, W) - 0.5 * av(dee(Hv), W))
        ru[:N] -= ((UFx - s(UFx, -1)) + (UFe - s(UFe, -W)))[:N]
        rv[:N] -= ((VFx - s(VFx, -1)) + (VFe - s(VFe, -W)))[:N]
        nt = (S2 // 512 + 1) * 512
        ru.view(-1)[S2:nt] = 0.0
        rv.view(-1)[S2:nt] = 0.0
        # vertical advection, fourth order, with the scheme's end levels
        k4 = lambda a: 9.0 / 16.0 * (a + s(a, S2)) - 1.0 / 16.0 * (s(a, -S2) + s(a, 2 * S2))
        h4 = lambda o: 9.0 / 16.0 * (self.W + s(self.W, o)) - 1.0 / 16.0 * (s(self.W, -o) + s(self.W, 2 * o))
        wu = h4(1)
        FU, FV = k4(u) * wu, k4(v) * h4(W)
        a, b = ru.clone(), rv.clone()
        a[2:N - 2] -= FU[3:N - 1] - FU[2:N - 2]
        b[2:N - 2] -= FV[3:N - 1] - FV[2:N - 2]
        b[1] -= 9.0 / 16.0 * (FV[1] + FV[2]) - 1.0 / 16.0 * (FV[1] + FV[3])
        f1 = (9.0 / 16.0 * (u[0] + u[1]) - 1.0 / 16.0 * u[2]) * wu[1]
        f0 = (9.0 / 16.0 * u[0] - 1.0 / 16.0 * u[1]) * wu[0]
        a[1] -= FU[2] - f1
        a[0] -= f1 - f0
        b[0] = b[1]
        for k in (N - 2, N - 1, N):
            a[k], b[k] = a[N - 3], b[N - 3]
        ok = self.inner & ~self.edge
        self.ru, self.rv = torch.where(ok, a, ru), torch.where(ok, b, rv)

    def zero_v_edges(self):
        v = self.v.view(self.N + 1, self.J, self.I)
        v[:-1, 1:-1, 0], v[:-1, 1:-1, -1], v[:-1, 0, :-1], v[:-1, -1, :-1] = 0.0, 0.0, 0.0, 0.0

    def sub(self, o, lam_dt):
        """Sub-diagonals -dt Akv/dz of the implicit viscosity: uses(k) the Akv level of row k."""
        dz = self.zr[1:] - self.zr[:-1]
        return lam_dt / (0.5 * (dz + self.s(dz, -o)))

    def step_uv(self, Zt_DU, Zt_DV, cff):
        """The reference's 3D momentum solve (first step: cff = 1)."""
        N, W = self.N, self.I
        out, elim = [], None
        uold, vold = self.u.clone(), self.v.clone()
        for d, o, x, r, Davg, met, node in ((0, 1, uold, self.ru, Zt_DU, self.onu, self.unode),
                                            (1, W, vold, self.rv, Zt_DV, self.omv, self.vnode)):
            Hx = 0.5 * (self.Hz + self.s(self.Hz, -o))
            Ak = 0.5 * (self.AKv + self.s(self.AKv, -o))
            SD = torch.zeros_like(Hx)
            SD[:N - 1] = self.sub(o, -self.dt) * Ak[:N - 1]
            c = cff * self.dt * (0.5 * (self.pm + _sh(self.pm, -o))) * (0.5 * (self.pn + _sh(self.pn, -o)))
            R = Hx * (x[:N] + c * r[:N])
            R[0] = 0.0
            D = Hx - SD
            D[1:] -= SD[:-1]
            D[0] = Hx[0] - 2.0 * SD[0]
            if d:       # rows that are u but not v points solve the eliminated u system again
                SD, D, R = (torch.where(node, a, b) for a, b in zip((SD, D, R), elim))
            for k in range(1, N):
                w = SD[k - 1] / D[k - 1]
                D[k] = D[k] - w * SD[k - 1]
                R[k] = R[k] - w * R[k - 1]
            elim = (SD, D, R)
            y = torch.zeros_like(R)
            y[N - 1] = R[N - 1] / D[N - 1]
            for k in range(N - 2, -1, -1):
                y[k] = (R[k] - SD[k] * y[k + 1]) / D[k]
            n = x.clone()
            n[:N] = torch.where(self.unode, y, x[:N])
            diff = ((x[:N] * Hx).sum(0) - Davg / met) / Hx.sum(0)
            n[:N] = torch.where(node, n[:N] - diff, n[:N])
            out.append(n)
        self.u, self.v = out
        bar = []
        for o, x, Davg, met in ((1, self.u, Zt_DU, self.onu), (W, self.v, Zt_DV, self.omv)):
            Hx = 0.5 * (self.Hz + self.s(self.Hz, -o))
            H, T = Hx.sum(0), Davg / met
            bar.append(T / H + ((Hx * x[:N]).sum(0) - T) / H)
        return bar

    def step_uv_coupled(self, Hz_old, su, sv, P, DU2, DV2):
        N, W, dt = self.N, self.I, self.dt
        bars = []
        for d, o, x, r, stress, D1, D2, Hf, m in ((0, 1, self.u, self.ru, su, P.DU, DU2, self.Hu, self.cu),
                                                  (1, W, self.v, self.rv, sv, P.DV, DV2, self.Hv, self.cv)):
            av = lambda a: 0.5 * (a + self.s(a, -o))
            Hx, Ak = av(self.Hz), av(self.AKv)
            SD = torch.zeros_like(Hx)
            SD[:N - 1] = self.sub(o, -dt) * Ak[1:N]
            c = dt * (0.5 * (self.pm + _sh(self.pm, -o))) * (0.5 * (self.pn + _sh(self.pn, -o)))
            R = av(Hz_old) * x[:N] + c * r[:N]
            D = Hx - SD
            D[1:] -= SD[:-1]
            R[0] = R[0] - dt * RDRG * x[0]
            R[N - 1] = R[N - 1] + dt * stress
            for k in range(1, N):
                w = SD[k - 1] / D[k - 1]
                D[k] = D[k] - w * SD[k - 1]
                R[k] = R[k] - w * R[k - 1]
            y = torch.zeros_like(R)
            y[N - 1] = R[N - 1] / D[N - 1]
            for k in range(N - 2, -1, -1):
                y[k] = (R[k] - SD[k] * y[k + 1]) / D[k]
            DC = (2.0 / (_sh(self.pm, -W) + self.pm) if d else 2.0 / (_sh(self.pn, -1) + self.pn)) * Hx
            Ds = DC.sum(0)
            y = y - ((DC * y).sum(0) - D1) / Ds
            bars.append((D1 / Ds, m))
            H = 0.5 * (Hf[:N] + y * DC)
            H = H - DC * (H.sum(0) - D2) / Ds
            x[:N] = torch.where(m, y, x[:N])
            Hf[:N] = torch.where(m, H, Hf[:N])
        return bars

    def pressure(self, T, S):
        N, W = self.N, self.I
        R0, T0, S0, Tc, Sc = EOS
        rho = (R0 - 1000.0) - R0 * Tc * (T - T0) + R0 * Sc * (S - S0)
        f1, f2, f3 = 0.5 * G / RHO0, 1000.0 * G / RHO0, 0.25 * G / RHO0
        for d, o, r, m in ((0, 1, self.ru, self.cu), (1, W, self.rv, self.cv)):
            p = lambda a: self.s(a, -o)
            met = 2.0 / (_sh(self.pm, -W) + self.pm) if d else 2.0 / (_sh(self.pn, -1) + self.pn)
            rp, zr, zp = p(rho), self.zr, p(self.zr)
            tw, tp = self.zw[N], _sh(self.zw[N], -o)
            Hs = 0.5 * (self.Hz + p(self.Hz))
            phi = f1 * (rho[N - 1] - rp[N - 1]) * ((tw - zr[N - 1]) + (tp - zp[N - 1])) \
                + (f2 + f1 * (rho[N - 1] + rp[N - 1])) * (tw - tp)
            for k in range(N - 1, -1, -1):
                if k < N - 1:
                    zf, zq = zr[k + 1] - zr[k], zp[k + 1] - zp[k]
                    g = 0.125 * ((zr[k] - zp[k]) + (zr[k + 1] - zp[k + 1])) * (zf - zq) / (zf * zq)
                    C1 = (1.0 + g) * (rho[k + 1] - rp[k + 1]) + (1.0 - g) * (rho[k] - rp[k])
                    C2 = (rho[k + 1] + rp[k + 1]) - (rho[k] + rp[k])
                    C3 = (zr[k + 1] + zp[k + 1]) - (zr[k] + zp[k])
                    C4 = (1.0 + g) * (zr[k + 1] - zp[k + 1]) + (1.0 - g) * (zr[k] - zp[k])
                    phi = phi + f3 * (C1 * C3 - C2 * C4)
                r[k] = torch.where(m, r[k] - Hs[k] * phi * met, r[k])
        return rho

    def tracer(self, t, Hz_old):
        N, W, s = self.N, self.I, self.s
        hu, hv = self.Hu[:N], self.Hv[:N]
        mn = self.pm * self.pn
        hu1, hv1 = s(self.Hu, 1)[:N], s(self.Hv, W)[:N]
        up = lambda f, o: torch.where(f > 0, s(t, -o), t)
        FX, FE = hu * up(hu, 1), hv * up(hv, W)
        FX1 = hu1 * torch.where(hu1 > 0, t, s(t, 1))
        FE1 = hv1 * torch.where(hv1 > 0, t, s(t, W))
        Wt = -torch.cumsum(mn * ((hu1 - hu) + (hv1 - hv)) + (self.Hz - Hz_old) / self.dt, 0)
        FC = Wt * t
        FC[:-1] = Wt[:-1] * torch.where(Wt[:-1] > 0, t[:-1], t[1:])
        div = mn * ((FX1 - FX) + (FE1 - FE)) + FC
        div[1:] -= FC[:-1]
        n = ((Hz_old * t - self.dt * div) / self.Hz).view(N, self.J, W).clone()
        n[:, 0], n[:, -1] = n[:, 1].clone(), n[:, -2].clone()
        n[:, :, 0], n[:, :, -1] = n[:, :, 1].clone(), n[:, :, -2].clone()
        return n

    def out(self):
        sh = (self.N + 1, self.J, self.I)
        return dict(u=self.u.reshape(-1), v=self.v.reshape(-1), ru=self.ru.reshape(-1), rv=self.rv.reshape(-1),
                    Huon=self.Hu.view(sh), Hvom=self.Hv.view(sh), W=self.W.view(sh), Hz=self.Hz.view(self.N, *sh[1:]),
                    z_w=self.zw.view(sh), z_r=self.zr.view(self.N, *sh[1:]))


def _exact_train(case, seed):
    d = _dev()
    Xb, Y, idx = _train_data(case, seed)
    X, Y = Xb.double().to(d), Y.double().to(d)
    p = torch.from_numpy(_net_params(seed)).double().to(d)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    sizes = [(IN, HID), (HID,), (HID, HID), (HID,), (HID, 16), (16,)]
    lr, b1, b2, eps = 1e-3, 0.9, 0.999, 1e-8
    for n, i in enumerate(idx, 1):
        W1, c1, W2, c2, W3, c3 = _split(p, sizes)
        x, y = X[i.long().to(d)], Y[i.long().to(d)]
        A1 = torch.relu(x @ W1 + c1)
        A2 = torch.relu(A1 @ W2 + c2)
        e = torch.zeros((x.shape[0], 16), dtype=torch.float64, device=d)
        e[:, :NOUT] = 2.0 * ((A2 @ W3 + c3)[:, :NOUT] - y) / (x.shape[0] * NOUT)
        d2 = (e @ W3.T) * (A2 > 0)
        d1 = (d2 @ W2.T) * (A1 > 0)
        g = torch.cat([t.reshape(-1) for t in (x.T @ d1, d1.sum(0), A1.T @ d2, d2.sum(0), A2.T @ e, e.sum(0))])
        m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
        p = p - lr * (m / (1 - b1 ** n)) / (torch.sqrt(v / (1 - b2 ** n)) + eps)
    return p.cpu().numpy()


def _split(p, sizes):
    out, o = [], 0
    for s in sizes:
        n = int(np.prod(s))
        out.append(p[o:o + n].reshape(s))
        o += n
    return out


def exact(case, seed):
    k = case["kind"]
    if k == "train":
        return _exact_train(case, seed)
    cfg, dtype = _config(case, seed), DT[case["dtype"]]
    if k == "ensemble":
        w1 = _weights(30)[0]
        out = []
        for c in cfg:
            b = _Basin2D(c, dtype)
            b.run(case["nsub"], w1)
            o = b.out()
            out.append((o["zeta"], o["ubar"], o["vbar"]))
        return out
    if k in ("barotropic", "open", "closure"):
        net = None
        if k == "closure":
            d = _dev()
            p = _split(torch.from_numpy(_net_params(seed)).double().to(d),
                       [(IN, HID), (HID,), (HID, HID), (HID,), (HID, 16), (16,)])
            mu, sd = (torch.from_numpy(a).double().to(d) for a in _norm(case, cfg))
            net = (p[0], p[1], p[2], p[3], p[4][:, :NOUT], p[5][:NOUT], mu, sd)
        b = _Basin2D(cfg, dtype, open_ext=_open_ext(case, seed) if k == "open" else None, net=net)
        b.run(case["nsub"], _weights(30)[0])
        return b.out()
    if k == "reference":
        b, w1 = _Reference2D(cfg), _weights(30)[0]
        for n in range(case["nsub"]):
            b.substep(w1[min(n, 256)])
        t2 = b.slot[2]
        return dict(zeta=torch.stack(b.z).reshape(3, b.J, b.I), ubar=b.u[t2], vbar=b.v[t2], Zt_avg1=b.Zt, DU_avg1=b.DU,
                    DV_avg1=b.DV)
    m = _Model3D(case, cfg, dtype)
    zeta0 = torch.from_numpy(np.array(cfg["zeta0"])).to(_dev()).reshape(-1)
    m.depths(zeta0)
    m.maxflux()
    m.omega()
    m.rhs()
    if k == "rhs3d":
        return dict(Huon=m.Hu.reshape(-1), Hvom=m.Hv.reshape(-1), W=m.W.reshape(-1), ru=m.ru.reshape(-1),
                    rv=m.rv.reshape(-1))
    w1, w2, nfast = _weights(case["ndtfast"])
    rn = (m.i > 0) & (m.j > 0)
    if k == "main3d":
        b = _Reference2D(cfg)
        for n in range(nfast + 1):
            b.substep(w1[n], zero_v=True)
        m.depths(b.Zt)
        ub, vb = m.step_uv(b.DU, b.DV, 1.0)
        t1, t2 = b.slot[1], b.slot[2]
        ub, vb = torch.where(m.unode, ub, b.u[t2]), torch.where(m.unode, vb, b.v[t2])
        m.zero_v_edges()
        m.omega()
        return dict(m.out(), Zt_avg1=b.Zt, DU_avg1=b.DU, DV_avg1=b.DV, zeta=torch.stack(b.z).reshape(3, b.J, b.I),
                    ubar=ub, vbar=vb)
    T, S = (torch.from_numpy(a).to(_dev(), dtype).double().reshape(m.N, m.S2) for a in _tracers(case, seed, cfg))
    rho = m.pressure(T, S)
    b = _Basin2D(cfg, dtype)
    for lv in (1, 2):
        b.put("zeta", lv, zeta0.to(dtype).double(), rn)
    zero = torch.zeros_like(zeta0)
    su, sv = (torch.from_numpy(np.array(cfg[n])).to(_dev()).reshape(-1) for n in ("sustr", "svstr"))
    inv = lambda a, o: 2.0 / (_sh(a, -o) + a)
    fr = []
    for o, r, x, st, mask in ((1, m.ru, m.u, su, m.cu), (m.I, m.rv, m.v, sv, m.cv)):
        fr.append(torch.where(mask, r[:m.N].sum(0) + (st - RDRG * x[0]) * inv(m.pm, o) * inv(m.pn, o), zero))
    cp = dict(rufrc=fr[0], rvfrc=fr[1], Fu=zero, Fv=zero, DU2=zero, DV2=zero)
    w = lambda i: w2[i - 1] if 1 <= i <= len(w2) else 0.0
    for iif in range(1, nfast + 2):
        cp["w2p"] = -w(2) / 12.0 if iif == 1 else (8.0 * w(iif) - w(iif + 1)) / 12.0
        cp["w2c"] = w(1) if iif == 1 else 5.0 / 12.0 * w(iif)
        b.rotate()
        b.substep(w1[iif - 1], first=iif == 1, cp=cp)
    Hz_old = m.Hz
    m.depths(b.Zt)
    bars = m.step_uv_coupled(Hz_old, su, sv, b, cp["DU2"], cp["DV2"])
    T, S = m.tracer(T, Hz_old), m.tracer(S, Hz_old)
    m.zero_v_edges()
    m.omega()
    for name, (x, mask) in zip(("ubar", "vbar"), bars):
        for lv in (1, 2):
            b.put(name, lv, x, mask)
    o = b.out()
    return dict(m.out(), Zt_avg1=b.Zt, DU_avg1=b.DU, DV_avg1=b.DV, zeta=o["zeta"], ubar=o["ubar"], vbar=o["vbar"], T=T,
                S=S, rho=rho.view(m.N, m.J, m.I), DU_avg2=cp["DU2"], DV_avg2=cp["DV2"])
