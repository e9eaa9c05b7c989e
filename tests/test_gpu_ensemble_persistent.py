"""Ensemble launches whose workgroups walk several tiles (a grid smaller than the tile count):
two workgroups a CU stay within a third of a workgroup per tile, and give its results."""
from __future__ import annotations

import sys

import pytest

from sailfish_amd import configs
from tests.test_gpu_ensemble import _diff

pytestmark = pytest.mark.gpu


def test_persistent_fp64_grid_keeps_two_workgroups_a_cu():
    """64 x 8 tiles, FP64, a grid of 512: 1.15 times one workgroup per tile measured; with one
    resident workgroup a CU it took 1.46."""
    import torch
    from sailfish_amd.ensemble import Member, PhysEnsemble
    print("[case] persistent ensemble", file=sys.stderr, flush=True)
    ms, out = [], []
    for sched in ((8, 1, 0), (8, 1, 512)):
        members = []
        for k in range(8):
            cfg = configs.ensemble_member(*((1024, 512), (768, 384))[k % 2], 0.05, 7 + k)
            cfg["dtfast"] = 5.0
            members.append(Member(cfg, dtype=torch.float64))
        ens = PhysEnsemble(members, torch.float64)
        ens.configure(*sched)
        ens.substep(True, 0.1)
        t = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(12):
                ens.substep(False, 0.1)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        ens.sync()
        ens.close()
        ms.append(sorted(t)[3])
        out.append(members)
    assert not _diff(*out)
    print(f"[persistent ensemble] {ms[1] / ms[0]}", file=sys.stderr, flush=True)
    assert ms[1] < 1.33 * ms[0], ms
