#!/usr/bin/env python3
"""Benchmark of the barotropic LF-AM3 substep on one MI355X.

Default workload (mode ``phys``): closed basin of 2048 x 1024 rho points, dx = 2 km,
seeded Gaussian-filtered bathymetry mapped to 200..4000 m, beta plane
f = 1e-4 + 2e-11 y, double-gyre wind tau_x = 0.1 cos(2 pi y / Ly), seeded 1 cm
free-surface noise, linear drag 3e-4 m/s, dt = 5 s; the ROMS 2D LF-AM3 substep
(predictor + corrector with C2 advection, Coriolis, stresses, drag) as ONE fused
launch (sf_phys_substep_fused).  Default precision: FP64 throughout, the reference's
precision (the form that matches the FP64 oracle bit for bit); ``--dtype f32`` runs
FP32 state and stencil arithmetic with the time averages in FP64.  The other
precision is measured too (``secondary``).  A "step" is one barotropic substep over
the whole grid; inputs are resident in HBM before timing starts.

Mode ``faithful``: the reference discretisation of nonlinear/step2d.py
(sf_step2d_substep, fused tile kernel) on the same grid, with the column-0/row-0
mask variant of computeMomentumPred.

Prints one JSON line.  The timed region is a HIP graph that holds the K substep
launches, each with its own arguments (slot rotation and averaging weight), one graph
per starting rotation so that consecutive replays continue the rotation; after at
least 150 ms of untimed replays, five replays are timed with HIP events on the replay
stream and ``ms_per_step`` is the median replay over K.  The same K launches issued one
by one are reported as ``config.ms_per_step_stream_launches``.  ``roofline`` is the
dominant kernel: algorithmic bytes per launch (the 29 fields of the substep) over its
mean launch time, which is the timed region's time per substep (the launches run back
to back; ``--no-graph`` times K stream launches and then 99 back-to-back launches
instead).
``cpu_baseline`` times the CPU oracle (C restatement, built with -O3 -march=native
on the machine that runs the benchmark) on a bounded number of substeps of the same
workload, on all the threads the process may use and on one.  ``secondary`` repeats the GPU measurement in the
other precision.  ``roofline.copy_GBs`` is the bandwidth of a plain 1 GiB device copy
on the same GPU (the practical streaming ceiling); ``large_grid`` repeats the FP32
kernel timing on a 4096 x 4096 basin whose working set is far beyond the 256 MB
last-level cache.  ``--calib-copy`` instead runs a plain device copy of known size
(the calibration run for the HBM byte counters).
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

HBM_PEAK_GBS = 8000.0
METRIC = "cell-steps/s + % HBM roofline; closure-coarse vs fine run at equal zeta RMSE"

# Algorithmic HBM bytes per rho point and substep, every field read or written once.
# physics substep (k_phys_fused):
#   reads : h, pm, pn, fomn, sustr, svstr, zeta/ubar/vbar at t0 and t1,
#           rzeta/rubar/rvbar at t0                                  (15 bulk)
#           Zt_avg1, DU_avg1, DV_avg1                                (3 FP64)
#   writes: zeta/ubar/vbar at t2, rzeta/rubar/rvbar at t1            (6 bulk)
#           Zt_avg1, DU_avg1, DV_avg1                                (3 FP64)
PHYS_BULK, PHYS_F64 = 21, 6
# The contract count of the same substep adds on_u and om_v (29 fields: 232 B FP64,
# 140 B FP32 state + FP64 averages); this kernel derives those two metric factors from
# pm and pn instead of reading them.  The roofline uses the contract count; the
# kernel's own read set (216 B / 132 B) is reported beside it.
PHYS_BULK_CONTRACT = 23
# timed region: REPS replays of K substeps after at least WARM_MS of untimed replays
REPS, WARM_MS = 5, 150.0
# reference-discretisation substep (k_step2d_fused):
#   reads : zeta_t1, zeta_t0, h, ubar_t1, vbar_t1, on_u, om_v, pm, pn,
#           rzeta_t0, rzeta_t2 (11 bulk), Zt/DU/DV_avg1 (3 FP64)
#   writes: zeta_t2, ubar_t2, vbar_t2, rzeta_t1 (4 bulk), averages (3 FP64)
# (the contract count, 168 B FP64; the kernel also writes rubar_t1, an observable array
# of the reference's predictor, which is not counted)
FAITHFUL_BULK, FAITHFUL_F64 = 15, 6


def _events(torch, n):
    return [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n)]


PHYS_KERNEL_SOURCES = ("sf_internal.h", "phys2d_fused_impl.h", "phys2d_fused.hip", "phys2d_fused_f32.hip")


def kernel_source_sha1() -> str:
    """SHA-1 over the sources of k_phys_fused (in PHYS_KERNEL_SOURCES order)."""
    import hashlib
    h = hashlib.sha1()
    for name in PHYS_KERNEL_SOURCES:
        h.update((ROOT / "sailfish_amd" / "csrc" / name).read_bytes())
    return h.hexdigest()


def measured_traffic(dtype_name):
    """HBM bytes per launch of k_phys_fused from the committed rocprofv3 FETCH_SIZE /
    WRITE_SIZE record (profiles/k_phys_fused_traffic.json), used only while the kernel
    source is the one that was profiled (same SHA-1); otherwise None."""
    rec_path = ROOT / "profiles" / "k_phys_fused_traffic.json"
    try:
        rec = json.loads(rec_path.read_text())
        if kernel_source_sha1() != rec["source_sha1"]:
            return None
        return int(rec[dtype_name]["hbm_bytes_per_launch"])
    except (OSError, KeyError, ValueError):
        return None


def phys_tile(precision, szI, szJ, tile_j=0):
    """[xi, eta] of the tile that sf_phys_substep_fused takes (tile_j = 0: its own choice)."""
    import ctypes as C
    from sailfish_amd import _lib
    from sailfish_amd.phys2d import _bind
    if tile_j:
        return [64, tile_j]
    a, b = C.c_int32(), C.c_int32()
    _lib.check(_bind().sf_phys_fused_tile(precision, 0, szI, szJ, C.byref(a), C.byref(b)), "sf_phys_fused_tile")
    return [a.value, b.value]


def run_phys_gpu(args, dtype_name, steps, warmup):
    import torch
    from sailfish_amd import configs
    from sailfish_amd.model2d import build_model
    from sailfish_amd.phys2d import PhysStepper

    dtype = torch.float64 if dtype_name == "f64" else torch.float32
    cfg = configs.basin2(args.szI, args.szJ, dx=args.dx)
    ct, GRID, OCEAN, _B = build_model(cfg, dtype=dtype, ndtfast=30)
    st = PhysStepper(GRID, OCEAN, rdrg=cfg["rdrg"], fused=True, tile_j=args.tile_j)
    tile_j = args.tile_j
    tile = phys_tile(st.precision, GRID.szI, GRID.szJ, tile_j)
    S2 = GRID.szI * GRID.szJ
    n = [0]

    def substep():
        ct.next2DTimeStep()
        OCEAN.cycleTimes2D()
        st.step(ct, OCEAN, first=(n[0] == 0))
        n[0] += 1

    for _ in range(max(warmup, 1)):
        substep()
    # the argument blocks of the three slot rotations, built once (three cycleTimes2D
    # bring the rotation back); launch k of the loop below uses rotation k % 3
    import ctypes as C
    from sailfish_amd import _lib
    blocks = []
    for _ in range(3):
        OCEAN.cycleTimes2D()
        blocks.append(st.fields(OCEAN))
    fn, prec, dt, sh = st.lib.sf_phys_substep_fused, st.precision, float(ct.dtfast), _lib.stream_handle()

    def launch(k):
        ct.next2DTimeStep()
        return fn(C.byref(blocks[k % 3]), prec, dt, 0, ct.cff1(), tile_j, sh)

    # the same K launches issued one by one from the host (reported for comparison)
    torch.cuda.synchronize()
    ev0, ev1 = _events(torch, 1)[0]
    ev0.record()
    rc = 0
    for k in range(steps):
        rc |= launch(k)
    ev1.record()
    torch.cuda.synchronize()
    _lib.check(rc, "sf_phys_substep_fused")
    ms_per_step_launched = ev0.elapsed_time(ev1) / steps
    done = steps

    if args.no_graph:
        for _ in range(done % 3):
            OCEAN.cycleTimes2D()
        n[0] += done
        ms_per_step, wall, ms_per_step_launched = ms_per_step_launched, 0.0, None
        nk = 99
        a, b = _events(torch, 1)[0]
        a.record()
        for k in range(nk):
            rc |= launch(done + k)
        b.record()
        torch.cuda.synchronize()
        _lib.check(rc, "sf_phys_substep_fused")
        kern_ms = a.elapsed_time(b) / nk
        finite = bool(torch.isfinite(OCEAN.zeta_t2).all()) and bool(torch.isfinite(OCEAN.ubar_t2).all())
        bulk = 8 if dtype_name == "f64" else 4
        bpp = PHYS_BULK_CONTRACT * bulk + PHYS_F64 * 8
        return dict(cfg=cfg, S2=S2, ms_per_step=ms_per_step, wall=wall, kern_ms=kern_ms, bpp=bpp,
                    bpp_read=PHYS_BULK * bulk + PHYS_F64 * 8,
                    achieved=bpp * S2 / (kern_ms * 1e-3) / 1e9, finite=finite,
                    zmax=float(OCEAN.zeta_t2.abs().max()), nk=nk, kernel="k_phys_fused",
                    entry="sf_phys_substep_fused", tile=tile, substeps=n[0] + nk)

    # the timed region: K substeps captured in HIP graphs, each node with its own
    # arguments (slot rotation and averaging weight of that substep).  Three graphs,
    # one per starting rotation, so that every replay continues the rotation where the
    # previous one left it, whatever K is: graph r holds substeps r, r+1, ... r+K-1 of
    # the rotation sequence.  Untimed replays warm the clocks (at least WARM_MS), then
    # REPS timed replays of exactly K substeps each; ms_per_step is the median replay
    # over K (HIP events on the replay stream).
    graphs = []
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    w_seq = []
    for _ in range(steps):
        ct.next2DTimeStep()
        w_seq.append(ct.cff1())
    with torch.cuda.stream(side):
        for r in range(3):
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                shc = _lib.stream_handle()
                for k in range(steps):
                    rc |= fn(C.byref(blocks[(r + k) % 3]), prec, dt, 0, w_seq[k], tile_j, shc)
            graphs.append(graph)
    torch.cuda.current_stream().wait_stream(side)
    _lib.check(rc, "sf_phys_substep_fused (capture)")
    pos = [done]

    def replay():
        graphs[pos[0] % 3].replay()
        pos[0] += steps

    torch.cuda.synchronize()
    t_w = time.perf_counter()
    nwarm = 0
    while nwarm < 2 or time.perf_counter() - t_w < WARM_MS * 1e-3:
        replay()
        nwarm += 1
        if nwarm % 4 == 0:
            torch.cuda.synchronize()
    torch.cuda.synchronize()
    rep_ms = []
    t0 = time.perf_counter()
    for _ in range(REPS):
        ev0, ev1 = _events(torch, 1)[0]
        ev0.record()
        replay()
        ev1.record()
        torch.cuda.synchronize()
        rep_ms.append(ev0.elapsed_time(ev1))
    wall = time.perf_counter() - t0
    rep_ms.sort()
    ms_per_step = rep_ms[len(rep_ms) // 2] / steps
    done = pos[0]
    for _ in range(done % 3):
        OCEAN.cycleTimes2D()
    n[0] += done
    del graphs
    # the graph replays the K launches back to back: the timed region's time per step is
    # the kernel's average launch duration (the kernel trace of the same replay agrees)
    kern_ms, nk = ms_per_step, steps
    finite = bool(torch.isfinite(OCEAN.zeta_t2).all()) and bool(torch.isfinite(OCEAN.ubar_t2).all())
    zmax = float(OCEAN.zeta_t2.abs().max())
    bulk = 8 if dtype_name == "f64" else 4
    bpp = PHYS_BULK * bulk + PHYS_F64 * 8
    bpp_contract = PHYS_BULK_CONTRACT * bulk + PHYS_F64 * 8
    achieved = bpp_contract * S2 / (kern_ms * 1e-3) / 1e9
    return dict(cfg=cfg, S2=S2, ms_per_step=ms_per_step, ms_per_step_launched=ms_per_step_launched, wall=wall,
                kern_ms=kern_ms, bpp=bpp_contract, bpp_read=bpp,
                achieved=achieved, finite=finite, zmax=zmax, nk=nk, kernel="k_phys_fused",
                entry="sf_phys_substep_fused", tile=tile, substeps=n[0],
                replays_ms=rep_ms, warm_replays=nwarm)


def run_large_grid_gpu(args):
    """The FP32 physics substep on a grid whose working set (2.2 GB) is far beyond the
    256 MB last-level cache: 4096 x 4096 basin2_analytic, 99 back-to-back launches."""
    import ctypes as C
    import torch
    from sailfish_amd import _lib, configs
    from sailfish_amd.model2d import build_model
    from sailfish_amd.phys2d import PhysStepper

    n = args.large
    cfg = configs.basin2_analytic(n, n, dx=args.dx)
    ct, GRID, OCEAN, _B = build_model(cfg, dtype=torch.float32, ndtfast=30)
    st = PhysStepper(GRID, OCEAN, rdrg=cfg["rdrg"], fused=True)
    for k in range(3):
        ct.next2DTimeStep()
        OCEAN.cycleTimes2D()
        st.step(ct, OCEAN, first=(k == 0))
    blocks = []
    for _ in range(3):
        OCEAN.cycleTimes2D()
        blocks.append(st.fields(OCEAN))
    fn, sh = st.lib.sf_phys_substep_fused, _lib.stream_handle()
    nk, rc = 99, 0
    torch.cuda.synchronize()
    a, b = _events(torch, 1)[0]
    a.record()
    for k in range(nk):
        ct.next2DTimeStep()
        rc |= fn(C.byref(blocks[k % 3]), st.precision, float(ct.dtfast), 0, ct.cff1(), 0, sh)
    b.record()
    torch.cuda.synchronize()
    _lib.check(rc, "sf_phys_substep_fused")
    ms = a.elapsed_time(b) / nk
    S2 = GRID.szI * GRID.szJ
    bpp = PHYS_BULK_CONTRACT * 4 + PHYS_F64 * 8
    return {"workload": f"basin2_analytic {n}x{n} (FP32 state, FP64 averages)", "points": S2, "kernel_ms": ms,
            "cell_steps_per_s": S2 / (ms * 1e-3), "achieved_GBs": bpp * S2 / (ms * 1e-3) / 1e9,
            "frac": bpp * S2 / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
            "finite_after_run": bool(torch.isfinite(OCEAN.zeta_t2).all())}


def copy_bandwidth():
    """Device-to-device copy of 1 GiB (read + write) with torch: the bandwidth a plain
    streaming kernel reaches on this GPU."""
    import torch
    n = 1 << 30
    src = torch.ones(n // 4, dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    dst.copy_(src)
    torch.cuda.synchronize()
    a, b = _events(torch, 1)[0]
    a.record()
    for _ in range(10):
        dst.copy_(src)
    b.record()
    torch.cuda.synchronize()
    ms = a.elapsed_time(b) / 10
    del src, dst
    return 2 * n / (ms * 1e-3) / 1e9


def run_faithful_gpu(args, dtype_name, steps, warmup):
    import torch
    from sailfish_amd import configs
    from sailfish_amd.model2d import build_model
    from sailfish_amd.step2d_fused import FusedStepper

    dtype = torch.float64 if dtype_name == "f64" else torch.float32
    cfg = configs.basin2(args.szI, args.szJ, dx=args.dx)
    ct, GRID, OCEAN, BOUNDARY = build_model(cfg, dtype=dtype, ndtfast=30, fix_q5=True)
    st = FusedStepper(GRID, BOUNDARY, dtype)
    S2 = GRID.szI * GRID.szJ

    def substep(parts=3):
        ct.next2DTimeStep()
        OCEAN.cycleTimes2D()
        st.step(ct, OCEAN, parts=parts)

    for _ in range(warmup):
        substep()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    ev0, ev1 = _events(torch, 1)[0]
    ev0.record()
    for _ in range(steps):
        substep()
    ev1.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms_per_step = ev0.elapsed_time(ev1) / steps
    # the tiled launch alone (the masked-points launch follows outside the events)
    nk = max(10, min(steps, 100))
    evs = _events(torch, nk)
    for a, b in evs:
        ct.next2DTimeStep()
        OCEAN.cycleTimes2D()
        a.record()
        st.step(ct, OCEAN, parts=1)
        b.record()
        st.step(ct, OCEAN, parts=2)
    torch.cuda.synchronize()
    kern_ms = sum(a.elapsed_time(b) for a, b in evs) / nk
    finite = bool(torch.isfinite(OCEAN.zeta_t2).all())
    bulk = 8 if dtype_name == "f64" else 4
    bpp = FAITHFUL_BULK * bulk + FAITHFUL_F64 * 8
    achieved = bpp * S2 / (kern_ms * 1e-3) / 1e9
    return dict(cfg=cfg, S2=S2, ms_per_step=ms_per_step, wall=wall, kern_ms=kern_ms, bpp=bpp,
                achieved=achieved, finite=finite, zmax=float(OCEAN.zeta_t2.abs().max()), nk=nk,
                kernel="k_step2d_fused", entry="sf_step2d_substep", tile=None, substeps=warmup + steps + nk)


def cpu_threads():
    """Threads of the CPU baseline: the cores this process may run on, capped by
    OMP_NUM_THREADS when the environment sets it (the CPU share of the machine)."""
    env = int(os.environ.get("SF_CPU_THREADS", "0") or 0)
    if env:
        return env
    n = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    omp = int(os.environ.get("OMP_NUM_THREADS", "0") or 0)
    return min(n, omp) if omp > 0 else n


_NATIVE = {}


def native_oracle():
    """The oracle's C restatement built for the machine that times it
    (gcc -O3 -march=native -ffp-contract=off -fopenmp), once per process, into a
    temporary directory; returns the use_library context of that build."""
    import tempfile
    from oracle import build, oracle as O
    if "path" not in _NATIVE:
        d = Path(tempfile.mkdtemp(prefix="sf_oracle_native_"))
        _NATIVE["path"] = build.build(verbose=False, out=d / "liboracle_native.so", opt="-O3",
                                      extra=["-march=native"])
    return O.use_library(_NATIVE["path"])


def _timed_runs(step, budget_s, runs=3):
    """One untimed warm-up step, then ``runs`` runs of n steps each (n sized so that
    the runs take about budget_s together); returns (median s per step, n)."""
    t0 = time.perf_counter()
    step()
    t1 = max(time.perf_counter() - t0, 1e-6)
    n = max(1, int(budget_s / runs / t1))
    per = []
    for _ in range(runs):
        t0 = time.perf_counter()
        for _ in range(n):
            step()
        per.append((time.perf_counter() - t0) / n)
    per.sort()
    return per[len(per) // 2], n


def _cpu_baseline(step_factory, units, unit, what, budget_s):
    """Median-of-3 rate of a CPU step on all threads and on one thread."""
    from oracle import oracle as O
    threads = cpu_threads()
    out = {}
    with native_oracle():
        for nt, share in ((threads, 0.4), (1, 0.6)):
            O.set_threads(nt)
            step = step_factory()
            sec, n = _timed_runs(step, budget_s * share)
            out[nt] = (units / sec, n)
        O.set_threads(threads)
    v_all, n_all = out[threads]
    v_one, n_one = out[1]
    return dict(value=v_all, unit=unit, cores=threads, kind="port",
                value_1core=v_one, nproc=os.cpu_count(),
                build="gcc -O3 -march=native -ffp-contract=off -fopenmp (built on this machine)",
                sample=f"{what}: median of 3 runs of {n_all} steps on {threads} OpenMP threads and of {n_one} "
                       f"steps on 1 thread, each after one warm-up step")


def run_cpu_phys(args, budget_s):
    """Physics-mode oracle (oracle/sf_oracle_phys.c, FP64, OpenMP) on the same grid."""
    from oracle import oracle_phys as OP
    from sailfish_amd import configs
    from sailfish_amd.mod_comptimes import CompTimes
    from sailfish_amd.mod_grid import update_metrics
    from sailfish_amd.set_weights import set_weights

    cfg = configs.basin2(args.szI, args.szJ, dx=args.dx)
    ct = CompTimes(cfg["dtfast"] * 30, 30)
    set_weights(ct)
    fomn = update_metrics(cfg["pm"], cfg["pn"], cfg["f"])["fomn"]
    o = OP.OPhys(cfg, fomn, rdrg=cfg["rdrg"])
    st = {"iif": o.run(1, cfg["dtfast"], ct.weight1)}      # first (Euler) substep

    def factory():
        def step():
            st["iif"] = o.run(1, cfg["dtfast"], ct.weight1, start_first=False, iif0=st["iif"])
        return step

    S2 = cfg["szI"] * cfg["szJ"]
    return _cpu_baseline(factory, S2, "cell-steps/s",
                         f"physics substeps of the {cfg['szI']}x{cfg['szJ']} basin (oracle C restatement, FP64)",
                         budget_s)


def run_cpu_faithful(args, budget_s):
    """Reference-discretisation oracle (one C function per reference kernel, OpenMP)."""
    from oracle import oracle as O
    from sailfish_amd import configs
    from sailfish_amd.mod_comptimes import CompTimes
    from sailfish_amd.mod_grid import update_metrics
    from sailfish_amd.set_weights import set_weights

    cfg = configs.basin2(args.szI, args.szJ, dx=args.dx)
    ct = CompTimes(cfg["dtfast"] * 30, 30)
    set_weights(ct)
    m = update_metrics(cfg["pm"], cfg["pn"], cfg["f"])
    g = O.OGrid(cfg["szI"], cfg["szJ"], 1, dict(h=cfg["h"], pm=cfg["pm"], pn=cfg["pn"], on_u=m["on_u"],
                                                   om_v=m["om_v"]), fix_q5=True)
    s = O.OState(g)
    for k in range(3):
        s.zeta[k][:] = cfg["zeta0"].ravel()
    b = O.OBoundary(g)
    t = O.OTimes(cfg["dtfast"], ct.weight1, ct.nfast)

    def factory():
        def step():
            O.main2d(t, g, s, b, 1)
        return step

    S2 = cfg["szI"] * cfg["szJ"]
    return _cpu_baseline(factory, S2, "cell-steps/s",
                         f"substeps of the {cfg['szI']}x{cfg['szJ']} basin (oracle C restatement of the reference "
                         "kernels, FP64)", budget_s)


def run_ensemble_gpu(args):
    """Ensemble workload: 64 members of the basin1 recipe with seeded uneven sizes,
    winds and noise; batched (one launch per substep, autotuned schedule, replayed
    from a HIP graph) vs looping the members one launch each."""
    import torch
    from sailfish_amd import autotune, configs
    from sailfish_amd.ensemble import LoopedMembers, Member, PhysEnsemble

    # the ensemble workload is specified with FP32 state and FP64 accumulators
    ens_dtype = "f32"
    dtype = torch.float32
    cfgs = configs.ensemble_configs(args.ens_members)
    members = [Member(c, dtype=dtype) for c in cfgs]
    ens = PhysEnsemble(members, dtype)
    pts = ens.points
    ct = members[0].ct
    ct.next2DTimeStep()
    ens.substep(True, ct.cff1())
    t0 = time.perf_counter()
    tuned = autotune.tune(ens, nsub=6, reps=2, use_cache=False)
    tune_s = time.perf_counter() - t0
    nsub = args.ens_steps - args.ens_steps % 3
    w = []
    for _ in range(3):
        ct.next2DTimeStep()
        w.append(ct.cff1())
    ens.capture(w)
    for _ in range(3):
        ens.replay()
    torch.cuda.synchronize()
    a, b = _events(torch, 1)[0]
    a.record()
    for _ in range(nsub // 3):
        ens.replay()
    b.record()
    torch.cuda.synchronize()
    ms_batched = a.elapsed_time(b) / nsub
    # the same substeps launched one at a time (no graph)
    a, b = _events(torch, 1)[0]
    a.record()
    for _ in range(30):
        ens.substep(False, w[0])
    b.record()
    torch.cuda.synchronize()
    ms_direct = a.elapsed_time(b) / 30
    ens.sync()
    finite = all(bool(torch.isfinite(m.OCEAN.zeta_t2).all()) for m in members)
    ens.close()
    looped = LoopedMembers(members)
    nl = max(3, min(30, nsub))
    for _ in range(3):
        looped.substep(False, w[0])
    torch.cuda.synchronize()
    a, b = _events(torch, 1)[0]
    a.record()
    for _ in range(nl):
        looped.substep(False, w[0])
    b.record()
    torch.cuda.synchronize()
    ms_looped = a.elapsed_time(b) / nl
    bulk = 8 if ens_dtype == "f64" else 4
    bpp = PHYS_BULK_CONTRACT * bulk + PHYS_F64 * 8
    return {
        "workload": f"{len(members)} basins (basin1 recipe, dx=5 km, dt=20 s), sizes drawn from "
                    "{256x128, 384x256, 512x256, 768x384, 1024x512} (seed 4), wind U[0.05,0.15] (seed 5)",
        "points": pts,
        "substeps_timed": nsub,
        "schedule": {"tile_j": tuned["tile_j"], "order": tuned["order"], "grid": tuned["grid"]},
        "autotune_s": tune_s,
        "batched_graph_ms_per_substep": ms_batched,
        "batched_graph_cell_steps_per_s": pts / (ms_batched * 1e-3),
        "batched_direct_ms_per_substep": ms_direct,
        "looped_ms_per_substep": ms_looped,
        "looped_cell_steps_per_s": pts / (ms_looped * 1e-3),
        "speedup_vs_looped": ms_looped / ms_batched,
        "hbm_frac_batched": bpp * pts / (ms_batched * 1e-3) / 1e9 / HBM_PEAK_GBS,
        "dtype": ens_dtype,
        "finite_after_run": finite,
    }


def run_closure_gpu(args):
    """Learned-closure workload: fine basin1 runs at 4x resolution (2042x1018 rho
    points, dx=312.5 m, dt=1.25 s) coarse-grained to 512x256 (dx=1.25 km, dt=5 s),
    2e6 samples, BF16-MFMA training, then 5000 coarse steps plain and with the
    closure against the coarse-grained fine run; speed of fine vs coarse+closure
    (FP32 and FP64, graph replays)."""
    import torch
    from sailfish_amd import closure as CL

    res = CL.run_experiment(dtype=torch.float64, log=lambda *a: print("[closure]", *a, file=sys.stderr, flush=True))
    mlp = res.pop("mlp")
    sp = CL.speed(mlp, dtype=torch.float32)
    sp64 = CL.speed(mlp, dtype=torch.float64, training=False)
    mlp.close()
    last = res["series"][-1]
    return {
        "workload": "basin1 recipe, fine 2042x1018 (dx 312.5 m, dt 1.25 s) -> coarse 512x256 (dx 1.25 km, "
                    "dt 5 s); 4 seeded training runs, 2e6 samples; evaluation: 5000 coarse steps of the "
                    "centred-bump configuration",
        "samples": res["samples"],
        "train_mse_normalised": [res["losses"][0], res["losses"][-1]],
        "train_s": res["train_s"],
        "target_rms_m_s2": res["target_rms"],
        "linear_r2": res["linear_r2"],
        "validation": res["validation"],
        "rmse_after_5000_steps": {"plain": last["plain"], "closure": last["closure"],
                                  "signal_max": last["signal"], "order": ["zeta_m", "ubar_m_s", "vbar_m_s"]},
        "selected_model": res["validation"]["selected"],
        "speed_fp32": sp,
        "speed_fp64": sp64,
        "experiment_s": res["total_s"],
    }


def run_3d_gpu(args):
    """Baroclinic 3D kernels (faithful reference discretisation, FP64) on a 1024 x 512
    basin1-recipe grid with 32 s-levels: rhs3d (Coriolis, horizontal and vertical
    advection) as one fused launch and as the three one-to-one kernels, set_maxflux and
    omega, each timed with HIP events on the launch stream.  A 3D cell-step = one (i, j, k) rho cell x one baroclinic step."""
    import numpy as np
    import torch
    from sailfish_amd import configs
    from sailfish_amd import mod_operators as ops
    from sailfish_amd.main3d import initial_depths
    from sailfish_amd.model2d import build_model3d

    szI, szJ, N = args.szI3, args.szJ3, args.N3
    cfg = configs.basin1(szI, szJ, dx=5e3)
    rng = np.random.Generator(np.random.PCG64(3))
    base = configs.gaussian_smooth(rng.standard_normal((szJ, szI)), 8.0)
    cfg["u0"] = 0.05 * base[None] * np.ones((N + 1, 1, 1))
    cfg["v0"] = 0.03 * base[None] * np.ones((N + 1, 1, 1))
    ct, GRID, OCEAN, BOUNDARY = build_model3d(cfg, N=N, ndtfast=40, dt=300.0, fix_q5=True)
    initial_depths(GRID, OCEAN)
    c = ops.ctx_of(GRID)
    BC = BOUNDARY.device_maps()["bcIdxFieldIdx2"]
    Huon, Hvom, W = OCEAN.Huon.reshape(-1), OCEAN.Hvom.reshape(-1), OCEAN.W.reshape(-1)
    Hz, z_w = GRID.Hz.reshape(-1), GRID.z_w.reshape(-1)
    S2 = GRID.szI * GRID.szJ
    grsz, bksz = (S2 // 512 + 1,), (512,)
    kern = {
        "set_maxflux": lambda: ops.set_maxflux(None, None, (OCEAN.u_t2, OCEAN.v_t2, Huon, Hvom, Hz), ctx=c),
        "omega": lambda: ops.omega(None, None, (W, OCEAN.u_t2, OCEAN.v_t2, Huon, Hvom, z_w, BC), ctx=c),
        "addCoriolis": lambda: ops.addCoriolis(grsz, bksz, (GRID.fomn.reshape(-1), OCEAN.u_t2, OCEAN.v_t2,
                                                            OCEAN.ru_t2, OCEAN.rv_t2, Hz), ctx=c),
        "horizontalAdvection": lambda: ops.horizontalAdvection(grsz, bksz, (OCEAN.u_t2, OCEAN.v_t2, Huon, Hvom,
                                                                            OCEAN.ru_t2, OCEAN.rv_t2, BC), ctx=c),
        "verticalAdvection": lambda: ops.verticalAdvection(grsz, bksz, (OCEAN.u_t2, OCEAN.v_t2, W, OCEAN.ru_t2,
                                                                        OCEAN.rv_t2, BC), ctx=c),
        "rhs3d_fused": lambda: ops.rhs3d_fused((GRID.fomn.reshape(-1), OCEAN.u_t2, OCEAN.v_t2, Huon, Hvom, W, Hz,
                                                OCEAN.ru_t2, OCEAN.rv_t2, BC), launch_threads=(S2 // 512 + 1) * 512,
                                               ctx=c),
    }
    # algorithmic FP64 bytes per 3D cell (fields read and/or written once); the fused
    # rhs3d reads u, v, Huon, Hvom, W, Hz and writes ru, rv
    fields = {"set_maxflux": 5, "omega": 4, "addCoriolis": 6, "horizontalAdvection": 6, "verticalAdvection": 5,
              "rhs3d_fused": 8}
    for f in kern.values():
        f()
    torch.cuda.synchronize()
    reps = 20
    out = {}
    cells = S2 * (N + 1)
    for name, f in kern.items():
        a, b = _events(torch, 1)[0]
        a.record()
        for _ in range(reps):
            f()
        b.record()
        torch.cuda.synchronize()
        ms = a.elapsed_time(b) / reps
        out[name] = {"ms": ms, "GB_s": fields[name] * 8 * cells / (ms * 1e-3) / 1e9}
    step = ("rhs3d_fused", "set_maxflux", "omega")      # the product path of one baroclinic step
    tot = sum(out[k]["ms"] for k in step)
    cells_int = S2 * N
    # FP32 bulk form of the same three kernels on the same state rounded to FP32
    u32, v32, Hz32, zw32 = (x.float() for x in (OCEAN.u_t2, OCEAN.v_t2, Hz, z_w))
    Hu32, Hv32, W32 = (torch.zeros(cells, dtype=torch.float32, device=u32.device) for _ in range(3))
    ru32, rv32 = torch.zeros_like(u32), torch.zeros_like(u32)
    kern32 = {
        "set_maxflux": lambda: ops.set_maxflux(None, None, (u32, v32, Hu32, Hv32, Hz32), ctx=c),
        "omega": lambda: ops.omega(None, None, (W32, u32, v32, Hu32, Hv32, zw32, BC), ctx=c),
        "rhs3d_fused": lambda: ops.rhs3d_fused((GRID.fomn.reshape(-1), u32, v32, Hu32, Hv32, W32, Hz32, ru32, rv32,
                                                BC), launch_threads=(S2 // 512 + 1) * 512, ctx=c),
    }
    for f in kern32.values():
        f()
    torch.cuda.synchronize()
    out32 = {}
    for name, f in kern32.items():
        a, b = _events(torch, 1)[0]
        a.record()
        for _ in range(reps):
            f()
        b.record()
        torch.cuda.synchronize()
        ms = a.elapsed_time(b) / reps
        out32[name] = {"ms": ms, "GB_s": fields[name] * 4 * cells / (ms * 1e-3) / 1e9}
    tot32 = sum(out32[k]["ms"] for k in step)
    res = {
        "workload": f"{szI}x{szJ}x{N} s-levels, basin1 recipe (dx 5 km), FP64, reference (faithful) 3D kernels",
        "kernels": out,
        "ms_rhs3d_maxflux_omega": tot,
        "cell_steps_per_s_3d": cells_int / (tot * 1e-3),
        "hbm_frac_3d": sum(fields[k] * 8 * cells for k in step) / (tot * 1e-3) / 1e9 / HBM_PEAK_GBS,
        "note": "rhs3d_fused (one launch) is the product path; addCoriolis / horizontalAdvection / "
                "verticalAdvection are the one-to-one reference kernels, timed for comparison",
        "fp32": {"kernels": out32, "ms_rhs3d_maxflux_omega": tot32, "cell_steps_per_s_3d": cells_int / (tot32 * 1e-3),
                 "hbm_frac_3d": sum(fields[k] * 4 * cells for k in step) / (tot32 * 1e-3) / 1e9 / HBM_PEAK_GBS,
                 "note": "FP32 bulk fields (2D metrics FP64, omega column sums FP64); bytes at 4 B per field"},
    }
    if not args.no_cpu:
        host = {k: x.detach().cpu().numpy().astype(np.float64).ravel() for k, x in
                dict(u=OCEAN.u_t2, v=OCEAN.v_t2, Huon=Huon, Hvom=Hvom, W=W, Hz=Hz, z_w=z_w).items()}
        res["cpu_baseline"] = run_cpu_3d(GRID, BOUNDARY, host, N, args.cpu_budget / 3)
    return res


def run_3d_step_gpu(args, dtype_name: str, coupled: bool):
    """The whole baroclinic step on the 1024 x 512 x 32 workload (configs.basin3: 40
    barotropic substeps per step of 300 s): the reference's loop body (main3d:
    set_maxflux, omega, set_zeta, rhs3d, 41 fused barotropic substeps, set_depth,
    step3d_UV, lateral BCs, omega) or the coupled form with the baroclinic pressure
    gradient and the tracer step (coupled3d).  Timed two ways: three steps issued from
    the host, and three steps captured in a HIP graph and replayed (median of 3 replays
    after 2 untimed ones; the three steps bring the slot rotation back).  A 3D
    cell-step = one (i, j, k) rho cell x one baroclinic step."""
    import torch
    from sailfish_amd import configs
    from sailfish_amd.main3d import Main3dState, baroclinic_step, initial_depths
    from sailfish_amd.model2d import build_model3d
    dtype = torch.float64 if dtype_name == "f64" else torch.float32
    cfg = configs.basin3(args.szI3, args.szJ3, args.N3)
    N = cfg["N"]
    ct, GRID, OCEAN, BOUNDARY = build_model3d(cfg, N=N, ndtfast=cfg["ndtfast"], dt=cfg["dt"], fix_q5=True,
                                              dtype=dtype)
    if coupled:
        from sailfish_amd.coupled3d import coupled_step, main3d_coupled
        st = main3d_coupled(ct, GRID, OCEAN, BOUNDARY, 1, tracers=True)     # includes the initial set_depth
        step = lambda: coupled_step(ct, GRID, OCEAN, BOUNDARY, st)
    else:
        m3 = Main3dState(GRID, OCEAN)
        initial_depths(GRID, OCEAN)
        step = lambda: baroclinic_step(ct, GRID, OCEAN, BOUNDARY, m3, fused=True)
        step()
    torch.cuda.synchronize()
    a, b = _events(torch, 1)[0]
    a.record()
    for _ in range(3):
        step()
    b.record()
    torch.cuda.synchronize()
    eager = a.elapsed_time(b) / 3
    res = {"ms_per_step_host_issued": eager}
    try:
        g = torch.cuda.CUDAGraph()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            with torch.cuda.graph(g, stream=s):
                for _ in range(3):
                    step()
        torch.cuda.current_stream().wait_stream(s)
        for _ in range(2):
            g.replay()
        torch.cuda.synchronize()
        times = []
        for _ in range(3):
            a, b = _events(torch, 1)[0]
            a.record()
            g.replay()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b) / 3)
        res["ms_per_step_graph"] = sorted(times)[1]
        res["graph_replays_ms_per_step"] = times
        ms = res["ms_per_step_graph"]
    except Exception as e:      # a capture that fails leaves the host-issued figure
        res["graph_error"] = f"{type(e).__name__}: {e}"
        ms = eager
    cells = N * GRID.szI * GRID.szJ
    res.update(ms_per_step=ms, cell_steps_per_s_3d=cells / (ms * 1e-3), dtype=dtype_name,
               finite_after_run=bool(torch.isfinite(OCEAN.u).all().item()),
               workload=(f"{GRID.szI}x{GRID.szJ}x{N}, 40 substeps per 300 s step, "
                         + ("coupled form + pressure gradient + tracers" if coupled else "reference loop body")))
    return res


def run_cpu_3d(GRID, BOUNDARY, host, N, budget_s):
    """The same 3D kernels (rhs3d with the reference's launch sizes, set_maxflux, omega)
    in the oracle's C restatement (FP64, OpenMP) on the same grid and state."""
    import numpy as np
    from oracle import oracle as O
    from oracle import oracle3d as O3

    hh = GRID.host
    g2 = O.OGrid(GRID.szI, GRID.szJ, 1, dict(h=hh["h"], pm=hh["pm"], pn=hh["pn"], on_u=hh["on_u"],
                                           om_v=hh["om_v"]))
    m = O3.OModel3(g2, N, hh["fomn"], hh["sc_r"], hh["sc_w"], hh["Cs_r"], hh["Cs_w"], GRID.hc, GRID.Vtransform,
                   BOUNDARY.zetaBC.bcIdxFieldIdx2, BOUNDARY.uvelBC.bcIdxFieldType,
                   BOUNDARY.vvelBC.bcIdxFieldType)
    m.u[2][:], m.v[2][:] = host["u"], host["v"]
    m.Huon[:], m.Hvom[:], m.W[:], m.z_w[:] = host["Huon"], host["Hvom"], host["W"], host["z_w"]
    m.Hz[:] = host["Hz"][:m.Hz.size]

    def factory():
        def step():
            L = O3.lib()
            m.rhs3d()
            L.sfo_set_maxflux(m.cp, O3.ptr(m.u[2]), O3.ptr(m.v[2]), O3.ptr(m.Huon), O3.ptr(m.Hvom), O3.ptr(m.Hz))
            L.sfo_omega(m.cp, O3.ptr(m.W), O3.ptr(m.Huon), O3.ptr(m.Hvom), O3.ptr(m.z_w), O3.ptr(m.BC))
        return step

    cells = GRID.szI * GRID.szJ * N
    return _cpu_baseline(factory, cells, "3D cell-steps/s",
                         f"rhs3d + set_maxflux + omega on {GRID.szI}x{GRID.szJ}x{N} (oracle C restatement, FP64)",
                         budget_s)


def calib_copy(args):
    """Plain device-to-device copy of 1 GiB, 5 times: the byte counters of this
    kernel calibrate FETCH_SIZE / WRITE_SIZE (2^30 bytes read and written each)."""
    import torch
    n = 1 << 30
    src = torch.ones(n // 4, dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(5):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"calib_copy_bytes": n, "launches": 5}))


def summary(r, dtype_name, steps, warmup):
    value = r["S2"] / (r["ms_per_step"] * 1e-3)
    return dict(value=value, ms_per_step=r["ms_per_step"], dtype=dtype_name, steps=steps, warmup=warmup,
                kernel=r["kernel"], kernel_ms=r["kern_ms"], bytes_per_point=r["bpp"],
                achieved_GBs=r["achieved"], frac=r["achieved"] / HBM_PEAK_GBS, finite_after_run=r["finite"])


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=500)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--mode", choices=["phys", "faithful"], default="phys")
    ap.add_argument("--dtype", choices=["f64", "f32"], default="f64")
    ap.add_argument("--tile-j", type=int, default=0)
    ap.add_argument("--szI", type=int, default=2048)
    ap.add_argument("--szJ", type=int, default=1024)
    ap.add_argument("--dx", type=float, default=2e3)
    ap.add_argument("--cpu-budget", type=float, default=15.0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-secondary", action="store_true")
    ap.add_argument("--calib-copy", action="store_true")
    ap.add_argument("--no-ensemble", action="store_true")
    ap.add_argument("--no-closure", action="store_true")
    ap.add_argument("--no-3d", action="store_true")
    ap.add_argument("--no-graph", action="store_true", help="time the headline as K stream launches (no HIP graph)")
    ap.add_argument("--large", type=int, default=4096, help="side of the beyond-cache grid (0: skip)")
    ap.add_argument("--szI3", type=int, default=1024)
    ap.add_argument("--szJ3", type=int, default=512)
    ap.add_argument("--N3", type=int, default=32)
    ap.add_argument("--ens-members", type=int, default=64)
    ap.add_argument("--ens-steps", type=int, default=498)
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: the benchmark runs on one GPU; --gpus {args.gpus} is not supported "
              "(the barotropic path would shard as row slabs with a 3-row halo exchange per substep)",
              file=sys.stderr)
        sys.exit(2)
    if args.calib_copy:
        calib_copy(args)
        return

    t_start = time.perf_counter()

    def progress(what):
        print(f"[bench] {what} done ({time.perf_counter() - t_start:.0f} s)", file=sys.stderr, flush=True)

    run = run_phys_gpu if args.mode == "phys" else run_faithful_gpu
    r = run(args, args.dtype, args.steps, args.warmup)
    progress(f"{args.mode} {args.dtype}")
    if not r["finite"]:
        raise SystemExit("bench.py: the headline state is not finite after the timed run")
    value = r["S2"] / (r["ms_per_step"] * 1e-3)
    if args.mode == "phys":
        workload = (f"ROMS 2D LF-AM3 barotropic substep (predictor+corrector, C2 advection, Coriolis, "
                    f"wind, linear drag), one fused launch; closed basin {args.szI}x{args.szJ} rho points, "
                    f"dx={args.dx/1e3:g} km, beta plane, dt=5 s")
    else:
        workload = (f"reference step2d discretisation (predictor+corrector), fused tile kernel; closed basin "
                    f"{args.szI}x{args.szJ} rho points, dx={args.dx/1e3:g} km, dt=5 s, column-0/row-0 mask")
    out = {
        "metric": METRIC,
        "value": value,
        "unit": "cell-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": r["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": args.dtype,
        "data": "synthetic",
        "config": {
            "workload": workload,
            "grid": [args.szI, args.szJ],
            "precision": "FP64" if args.dtype == "f64" else "FP32 state, FP64 time averages",
            "entry": r["entry"],
            "tile": r["tile"],
            "finite_after_run": r["finite"],
            "max_abs_zeta_after_run": r["zmax"],
            "substeps_run": r["substeps"],
            "timed_as": (f"median of {REPS} replays of a HIP graph holding the K substep launches, each with "
                         f"its own arguments, after >= {WARM_MS:g} ms of untimed replays"
                         if r.get("ms_per_step_launched") else "K stream launches"),
            "replay_ms": r.get("replays_ms"),
            "ms_per_step_stream_launches": r.get("ms_per_step_launched"),
        },
        "roofline": {
            "bound": "hbm",
            "achieved": r["achieved"],
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": r["achieved"] / HBM_PEAK_GBS,
            "traffic": measured_traffic(args.dtype) if args.mode == "phys" and args.szI == 2048
            and args.szJ == 1024 and args.tile_j in (0, 8) else None,
            "kernel": r["kernel"],
            "kernel_ms": r["kern_ms"],
            "bytes_per_point": r["bpp"],
            "bytes_per_point_kernel_reads": r.get("bpp_read"),
            "frac_at_kernel_reads": (r.get("bpp_read") or r["bpp"]) * r["S2"] / (r["kern_ms"] * 1e-3) / 1e9
            / HBM_PEAK_GBS,
            "points_per_launch": r["S2"],
            "launches_timed": r["nk"],
        },
    }
    out["roofline"]["copy_GBs"] = copy_bandwidth()
    if args.large and args.mode == "phys":
        out["large_grid"] = run_large_grid_gpu(args)
        progress("large grid")
    if not args.no_secondary:
        other = "f32" if args.dtype == "f64" else "f64"
        s2 = run(args, other, min(args.steps, 200), args.warmup)
        out["secondary"] = summary(s2, other, min(args.steps, 200), args.warmup)
        progress(f"secondary {other}")
    if not args.no_secondary and args.mode == "phys":
        # the reference discretisation (faithful mode, FP64, bitwise equal to the oracle) on
        # the same grid, with the column-0/row-0 mask variant
        # warm-up 5 + 40 timed + 40 single-launch substeps: the reference discretisation
        # stays finite for ~120 substeps at dt = 5 s on this grid
        fa = run_faithful_gpu(args, "f64", 40, 5)
        out["faithful"] = summary(fa, "f64", 40, 5)
        out["faithful"]["workload"] = ("reference step2d discretisation (nonlinear/step2d.py), fused tile kernel, "
                                       f"{args.szI}x{args.szJ}, FP64")
        if not args.no_cpu:
            out["faithful"]["cpu_baseline"] = run_cpu_faithful(args, args.cpu_budget / 3)
        progress("faithful f64")
    if not args.no_ensemble and args.mode == "phys":
        out["ensemble"] = run_ensemble_gpu(args)
        progress("ensemble")
    if not args.no_closure and args.mode == "phys":
        out["closure"] = run_closure_gpu(args)
        progress("closure")
    if not args.no_3d and args.mode == "phys":
        out["baroclinic_3d"] = run_3d_gpu(args)
        progress("3d")
        out["baroclinic_3d"]["whole_step"] = {
            f"{'coupled' if cp else 'reference'}_{d}": run_3d_step_gpu(args, d, cp)
            for cp in (False, True) for d in ("f64", "f32")}
        progress("3d whole step")
    if not args.no_cpu:
        out["cpu_baseline"] = (run_cpu_phys if args.mode == "phys" else run_cpu_faithful)(args, args.cpu_budget)
        progress("cpu baseline")
    print(json.dumps(out))


if __name__ == "__main__":
    main()
