"""phys2d.issue_substeps on the CPU: counters, weights and view rotation as a loop of single
substeps leaves them, for every remainder of the slot rotation and when a substep fails."""
from __future__ import annotations

import types

import pytest

from sailfish_amd import _lib
from sailfish_amd.mod_comptimes import CompTimes
from sailfish_amd.mod_ocean import T_OCEAN
from sailfish_amd.phys2d import issue_substeps


def _model():
    ct = CompTimes(dt=0.3, ndtfast=3)
    ct.weight1[:5] = [0.1, 0.2, 0.3, 0.25, 0.15]
    return ct, T_OCEAN(types.SimpleNamespace(N=1, M=3, L=3, device="cpu"), with3d=False)


def _loop(nsub):
    ct, oc = _model()
    w = []
    for _ in range(nsub):
        ct.next2DTimeStep()
        oc.cycleTimes2D()
        w.append(ct.cff1())
    return ct, oc, w


@pytest.mark.parametrize("nsub", [0, 1, 2, 3, 7])
def test_counters_and_views(nsub):
    ct, oc = _model()
    got = {}

    def issue(n, w, cl, done):
        got.update(n=n, w=list(w)[:n], cl=list(cl)[:n])
        done.value = n
        return _lib.SF_OK

    issue_substeps(ct, oc, nsub, "x", issue, clamp=lambda t: 2.0 * t)
    ct0, oc0, w0 = _loop(nsub)
    assert got["n"] == nsub and got["w"] == w0
    assert (ct.iif, ct.time2D) == (ct0.iif, ct0.time2D)
    assert not nsub or got["cl"][-1] == 2.0 * ct0.time2D
    for lev in ("t0", "t1", "t2"):
        assert oc.slot_of("vbar", lev) == oc0.slot_of("vbar", lev)


@pytest.mark.parametrize("done_before", [0, 1, 4])
def test_failure_stops_where_the_loop_would(monkeypatch, done_before):
    ct, oc = _model()

    def issue(n, w, cl, done):
        done.value = done_before
        return 1

    def check(rc, what):
        if rc:
            raise _lib.SailfishError(what)

    monkeypatch.setattr(_lib, "check", check)
    with pytest.raises(_lib.SailfishError):
        issue_substeps(ct, oc, 6, "x", issue)
    ct0, oc0, _w = _loop(done_before + 1)
    assert (ct.iif, ct.time2D) == (ct0.iif, ct0.time2D)
    assert oc.slot_of("zeta", "t2") == oc0.slot_of("zeta", "t2")
