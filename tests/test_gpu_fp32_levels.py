"""FP32 instances of the on-chip 3D momentum steps at the edges of their level counts (up to
16, 24, 32, 40, 48 and 64 levels).

- The coupled step against its scratch form, bit for bit: that form takes grids whose N + 1
  levels pass 4 GiB.  Inputs vary along xi and with the level only, so a grid of twelve rows,
  solved on chip, has every value of the large one.
- The reference's step3d_UV against FP64, within the bounds of the shallow columns."""
from __future__ import annotations

import ctypes as C
import sys

import pytest

from sailfish_amd import _lib
from tests.test_gpu_large_grids import SZI, _ctx, _need, _rows, _same
from tests.test_gpu_step3d import test_fp32_bulk_step3d_uv_against_fp64 as uv_case

pytestmark = pytest.mark.gpu

LEVELS = [24, 25, 33, 40, 41, 48, 49, 64]


@pytest.mark.parametrize("N", LEVELS)
def test_coupled_fp32_on_chip_equals_scratch(N):
    import torch
    from sailfish_amd.coupled3d import _bind, sf_uv_coupled
    print(f"[case] coupled FP32 levels {N}", file=sys.stderr, flush=True)
    _need(torch, 110)
    lib, f32, f64, out = _bind(), torch.float32, torch.float64, []
    for szJ in (12, 2 ** 32 // (4 * (N + 1) * SZI) + 2):
        r = lambda lo, hi, seed, n=N, t=f32: _rows(torch, szJ, n, lo, hi, seed, t)
        u, v, ru, ru1, ru2 = r(-1, 1, 1), r(-1, 1, 2), r(-1, 1, 3), r(-1, 1, 4), r(-1, 1, 5)
        ku, kv, Ho, Hz, Ak, z_r = r(0, 0, 0), r(0, 0, 0), r(9, 11, 6), r(9, 11, 7), r(1e-3, 2e-3, 8), r(0, 1, 9)
        for k in range(N):
            z_r[k] += 10.0 * k
        Hu, Hv, scratch = r(-50, 50, 10), r(-50, 50, 11), [torch.empty_like(u) for _ in range(3)]
        metric, D1, D2, st = (r(lo, hi, seed, 1, f64) for lo, hi, seed in ((.9, 1.1, 12), (-99, 99, 13), (-99, 99, 14),
                                                                         (-1, 1, 15)))
        ub, vb = torch.zeros((2, 1, szJ, SZI), dtype=f32, device="cuda")
        q = lambda *t: [x.data_ptr() for x in t]
        a = sf_uv_coupled(*q(u, v, ru, ru, ru1, ru1, ru2, ru2, ku, kv, ub, vb, ub, vb, Ho, Hz, Ak, z_r, D1, D1, D2, D2,
                             Hu, Hv, st, st), 3e-4, 2, *q(*scratch))
        ctx = _ctx(torch, szJ, N, metric)
        _lib.check(lib.sf_step3d_uv_coupled(ctx, _lib.SF_FP32, C.byref(a), 1.0, 60.0, _lib.stream_handle()),
                   "sf_step3d_uv_coupled")
        torch.cuda.synchronize()
        _lib.load().sf_ctx_destroy(ctx)
        out.append((u, v, Hu, Hv, ku, kv, ub, vb))
        del ru, ru1, ru2, Ho, Hz, Ak, z_r, scratch, metric, D1, D2, st
    names = ("u", "v", "Huon", "Hvom", "ru_keep", "rv_keep", "ubar", "vbar")
    bad = [(n, _same(b, s)) for n, s, b in zip(names, *out)]
    del u, v, Hu, Hv, ku, kv, ub, vb, out
    torch.cuda.empty_cache()
    assert not any(x for _n, x in bad), bad


@pytest.mark.parametrize("N", LEVELS)
def test_step3d_uv_fp32(N):
    uv_case(40, 30, N)
