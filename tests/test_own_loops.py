"""A caller's own counter, state or step class (or a method replaced on one object) is stepped
substep by substep: next2DTimeStep, cycleTimes2D, substep, in that order; only the
framework's own go through the native loop.  On the CPU, with a library that records calls."""
from __future__ import annotations

import types

import pytest
import torch

from sailfish_amd import _lib, phys2d, step2d_fused
from sailfish_amd.coupled3d import CoupledState, _coupled_substeps
from sailfish_amd.main2d import barotropic_loop, main2d
from sailfish_amd.mod_comptimes import CompTimes
from sailfish_amd.mod_ocean import T_OCEAN
from sailfish_amd.phys2d import PhysStepper, run_phys
from sailfish_amd.step2d_fused import FusedStepper

GRID = types.SimpleNamespace(N=1, M=3, L=3, szI=4, szJ=4, device="cpu")


class Counter(CompTimes):
    def next2DTimeStep(self):
        super().next2DTimeStep()
        self.log.append("next")


class State(T_OCEAN):
    def cycleTimes2D(self):
        super().cycleTimes2D()
        self.log.append("cycle")


class Properties(T_OCEAN):
    """A state that keeps one view under another name."""

    @property
    def zeta_t0(self):
        return self.hidden

    @zeta_t0.setter
    def zeta_t0(self, v):
        self.hidden = v


class Wind(PhysStepper):
    def fields(self, OCEAN):
        self.log.append("fields")
        return super().fields(OCEAN)


class Step(FusedStepper):
    def step(self, compTimes, OCEAN, zero_vbar=False, stream=None, parts=3):
        self.log.append("substep")


class Couple(CoupledState):
    def couple_fields(self, n, iif, weight2):
        self.log.append("couple")
        return super().couple_fields(n, iif, weight2)


class Lib:
    """Records the native calls; every one succeeds."""

    def __init__(self, log):
        self.log = log

    def __getattr__(self, name):
        def call(*args):
            if name.endswith("_run"):
                args[-1]._obj.value = 0
                self.log.append("native")
            else:
                self.log.append("substep")
            return _lib.SF_OK
        return call


@pytest.fixture
def log(monkeypatch):
    monkeypatch.setattr(_lib, "stream_handle", lambda stream=None: None)
    return []


def _counter(log, cls=CompTimes):
    ct = cls(dt=0.4, ndtfast=4)
    ct.nfast = 3
    ct.log = log
    return ct


def _state(log, cls=T_OCEAN):
    oc = cls(GRID, with3d=False)
    oc.log = log
    return oc


def _stepper(log, cls=PhysStepper):
    st = cls.__new__(cls)
    st.log, st.lib = log, Lib(log)
    st.static = {k: torch.zeros(16, dtype=torch.float64) for k in ("h", "pm", "pn", "fomn", "sustr", "svstr")}
    st.szI, st.szJ, st.g, st.rdrg, st.open_edges, st.fused, st.tile_j = 4, 4, 10.0, 0.0, 0, True, 0
    st.scratch, st.precision = [], _lib.SF_FP64
    return st


def _fused(log, cls=FusedStepper):
    st = cls.__new__(cls)
    st.log, st.lib, st.dtype, st.precision = log, Lib(log), torch.float64, _lib.SF_FP64
    st.ctx = types.SimpleNamespace(handle=None)
    st.grid_fields = {k: torch.zeros(16, dtype=torch.float64) for k in ("h", "on_u", "om_v", "pm", "pn")}
    return st


def _coupled(log, cls=CoupledState):
    st = cls.__new__(cls)
    st.log, st.lib, st.fused, st.tile_j = log, Lib(log), True, 0
    z = lambda: torch.zeros(16, dtype=torch.float64)
    st.rufrc, st.rvfrc, st.DU_avg2, st.DV_avg2 = z(), z(), z(), z()
    st.Fu, st.Fv = [z() for _ in range(3)], [z() for _ in range(3)]
    st.stepper = _stepper(log)
    return st


def _replace(obj, name, word):
    """Put a logging version of a method on the object itself."""
    bound = getattr(obj, name)

    def logged(*a, **k):
        r = bound(*a, **k)
        obj.log.append(word)
        return r
    setattr(obj, name, logged)
    return obj


CASES = {
    "own": lambda g: (_counter(g), _state(g), _stepper(g), ["native"]),
    "counter": lambda g: (_counter(g, Counter), _state(g), _stepper(g), ["next", "substep"]),
    "counter on the object": lambda g: (_replace(_counter(g), "next2DTimeStep", "next"), _state(g), _stepper(g),
                                        ["next", "substep"]),
    "state": lambda g: (_counter(g), _state(g, State), _stepper(g), ["cycle", "substep"]),
    "state on the object": lambda g: (_counter(g), _replace(_state(g), "cycleTimes2D", "cycle"), _stepper(g),
                                      ["cycle", "substep"]),
    "fields": lambda g: (_counter(g), _state(g), _stepper(g, Wind), ["fields", "substep"]),
    "step on the object": lambda g: (_counter(g), _state(g), _replace(_stepper(g), "step", "step"),
                                     ["substep", "step"]),
}


@pytest.mark.parametrize("case", CASES)
def test_run_phys(log, case):
    ct, oc, st, unit = CASES[case](log)
    slot = oc.slot_of("zeta", "t2")
    run_phys(ct, GRID, oc, 4, st)
    assert log == (unit if case == "own" else unit * 4)
    assert ct.iif == 4 and oc.slot_of("zeta", "t2") == (slot + 4) % 3


@pytest.mark.parametrize("loop", ["main2d", "barotropic_loop"])
@pytest.mark.parametrize("case", ["own", "counter", "state", "step", "state on the object"])
def test_step2d(log, loop, case):
    ct = _counter(log, Counter if case == "counter" else CompTimes)
    oc = _state(log, State if case == "state" else T_OCEAN)
    if case == "state on the object":
        _replace(oc, "cycleTimes2D", "cycle")
    grid = types.SimpleNamespace(**vars(GRID), _sf_fused=_fused(log, Step if case == "step" else FusedStepper))
    if loop == "main2d":
        main2d(ct, grid, oc, None, 4, fused=True)
    else:
        barotropic_loop(ct, grid, oc, None, fused=True)
    unit = dict(own=["native"], counter=["next", "substep"], state=["cycle", "substep"], step=["substep"])
    unit["state on the object"] = unit["state"]
    assert log == (unit[case] if case == "own" else unit[case] * 4)


@pytest.mark.parametrize("case", ["own", "counter", "state", "couple", "stepper"])
def test_coupled(log, case):
    ct = _counter(log, Counter if case == "counter" else CompTimes)
    oc = _state(log, State if case == "state" else T_OCEAN)
    st = _coupled(log, Couple if case == "couple" else CoupledState)
    if case == "stepper":
        st.stepper = _stepper(log, Wind)
    oc.Zt_avg1 += 1.0
    _coupled_substeps(ct, oc, st, st.lib, None)
    unit = dict(counter=["next", "substep"], state=["cycle", "substep"], couple=["couple", "substep"],
                stepper=["fields", "substep"])
    assert log == (["native"] if case == "own" else unit[case] * 4)
    assert not oc.Zt_avg1.any()


def test_views_of_a_subclass_rotate(log):
    oc = _state(log, Properties)
    a, b, c = oc.zeta_t0, oc.zeta_t1, oc.zeta_t2
    oc.cycleTimes2D()
    assert oc.zeta_t0 is b and oc.zeta_t1 is c and oc.zeta_t2 is a


def test_method_replaced_on_the_class(log, monkeypatch):
    plain = CompTimes.next2DTimeStep
    monkeypatch.setattr(CompTimes, "next2DTimeStep", lambda self: (plain(self), log.append("next")))
    ct, oc, st = _counter(log), _state(log), _stepper(log)
    run_phys(ct, GRID, oc, 3, st)
    assert log == ["next", "substep"] * 3


@pytest.mark.parametrize("nsub", [-1, -2, -5])
def test_negative_counts_do_nothing(log, nsub):
    ct, oc = _counter(log), _state(log)
    grid = types.SimpleNamespace(**vars(GRID), _sf_fused=_fused(log))
    slots = [oc.slot_of("zeta", f"t{k}") for k in range(3)]
    run_phys(ct, GRID, oc, nsub, _stepper(log))
    main2d(ct, grid, oc, None, nsub, fused=True)
    step2d_fused.step2d_run(ct, grid, oc, None, nsub)
    grid._sf_fused.run(ct, oc, nsub)
    phys2d.issue_substeps(ct, oc, nsub, "x", lambda *a: _lib.SF_ERR_ARG)
    assert (ct.iif, ct.time2D) == (0, 0.0) and not log
    assert [oc.slot_of("zeta", f"t{k}") for k in range(3)] == slots


class RunLib(Lib):
    """The native run: records (first, count) of each call."""

    def __getattr__(self, name):
        def call(*args):
            if name == "sf_phys_run":
                self.log.append((args[9], args[11]))
                args[-1]._obj.value = args[11]
            else:
                self.log.append((None, args[7]))
                args[-1]._obj.value = args[7]
            return _lib.SF_OK
        return call


@pytest.mark.parametrize("nsub", [3071, 3072, 3073, 20000])
def test_long_runs_go_in_bounded_calls(log, nsub):
    """A native call keeps signals waiting and holds its weights: a long run takes several, and
    its memory does not grow with it."""
    import tracemalloc
    for run in ("phys", "step2d"):
        log.clear()
        ct, oc = _counter(log), _state(log)
        slot = oc.slot_of("zeta", "t2")
        st, fs = _stepper(log), _fused(log)
        st.lib, fs.lib = RunLib(log), RunLib(log)
        grid = types.SimpleNamespace(**vars(GRID), _sf_fused=fs)
        tracemalloc.start()
        if run == "phys":
            run_phys(ct, GRID, oc, nsub, st)
        else:
            main2d(ct, grid, oc, None, nsub, fused=True)
        peak = tracemalloc.get_traced_memory()[1]
        tracemalloc.stop()
        counts = [c for _f, c in log]
        assert sum(counts) == nsub and max(counts) <= 3072 and all(c % 3 == 0 for c in counts[:-1])
        assert run == "step2d" or [f for f, _c in log] == [1] + [0] * (len(log) - 1)
        assert ct.iif == nsub and oc.slot_of("zeta", "t2") == (slot + nsub) % 3
        assert peak < 300_000, peak
