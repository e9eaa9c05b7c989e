"""3D kernels on grids whose levels pass 4 GiB or 2^30 points.  Every input varies along xi
and with the level only, so rows away from the south and north edges repeat, and a grid of
twelve rows gives every value: bit for bit."""
from __future__ import annotations

import ctypes as C
import sys

import pytest

from sailfish_amd import _lib

pytestmark = pytest.mark.gpu

SZI = 65536


def _ctx(torch, szJ, N, metric):
    d = _lib.sf_grid_desc(SZI, szJ, N, 0, *[metric.data_ptr()] * 4)
    h = C.c_void_p()
    _lib.check(_lib.load().sf_ctx_create(C.byref(d), C.byref(h)), "sf_ctx_create")
    return h


def _need(torch, gib):
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < gib * 2 ** 30:
        pytest.skip(f"needs {gib} GiB of GPU memory")


def _rows(torch, szJ, levels, lo, hi, seed, dtype):
    """A field of `levels` levels with the same row of values in lo .. hi at every eta."""
    g = torch.Generator().manual_seed(seed)
    row = lo + (hi - lo) * torch.rand((levels, 1, SZI), generator=g, dtype=torch.float64)
    t = torch.empty((levels, szJ, SZI), dtype=dtype, device="cuda")
    t.copy_(row.to(dtype).cuda().expand(levels, szJ, SZI))
    return t


def _same(big, small):
    """Rows of the big grid against those of the small one: six at either edge, the rest alike."""
    bad = []
    for k in range(big.shape[0]):
        if not bool((big[k, :6] == small[k, :6]).all()) or not bool((big[k, -6:] == small[k, -6:]).all()):
            bad.append((k, "edges"))
        for r in range(6, big.shape[1] - 6, 2048):
            if not bool((big[k, r:min(r + 2048, big.shape[1] - 6)] == small[k, 5]).all()):
                bad.append((k, r))
    return bad


@pytest.mark.parametrize("dt,szJ", [("f64", 8200), ("f32", 16400)])
def test_step3d_uv_levels_past_4_gib(dt, szJ):
    """tmpU, tmpV alias u, v, as the driver passes them."""
    import torch
    print(f"[case] step3d_UV level of {SZI} x {szJ} {dt}", file=sys.stderr, flush=True)
    _need(torch, 150)
    T = torch.float64 if dt == "f64" else torch.float32
    N, out = 4, []
    for sz in (12, szJ):
        r = lambda lo, hi, seed, n=N, t=T: _rows(torch, sz, n, lo, hi, seed, t)
        u, v, ru, Hz, Akv = r(-1, 1, 1), r(-1, 1, 2), r(-1, 1, 3), r(9, 11, 4), r(1e-3, 2e-3, 5)
        z_r = r(0, 1, 6)
        for k in range(N):
            z_r[k] += 10.0 * k
        metric, D = r(0.9, 1.1, 7, 1, torch.float64), r(-1, 1, 8, 1, torch.float64)
        ub, vb = torch.zeros((2, 1, sz, SZI), dtype=T, device="cuda")
        ctx = _ctx(torch, sz, N, metric)
        p = [t.data_ptr() for t in (u, v, ru, ru, ub, vb, ub, vb, Hz, Akv, z_r, D, D, u, v)]
        _lib.call("sf_step3d_uv" + ("" if dt == "f64" else "_f32"), ctx, *p, 5, 0, 1.0, 10.0,
                  *[ru.data_ptr()] * 3, _lib.stream_handle())
        torch.cuda.synchronize()
        _lib.load().sf_ctx_destroy(ctx)
        out.append((u, v, ub, vb))
        del ru, Hz, Akv, z_r, metric, D
    bad = [(n, _same(b, a)) for n, a, b in zip(("u", "v", "ubar", "vbar"), *out)]
    del u, v, ub, vb, out
    torch.cuda.empty_cache()
    assert not any(x for _n, x in bad), bad


def test_split_columns_past_2_30_points():
    """set_maxflux, omega, pressure gradient and tracer step of more than 2^30 columns (four
    threads to a column pass what one launch takes along x), FP32."""
    import torch
    from sailfish_amd.baroclinic import _bind
    szJ, N = 16400, 4
    print(f"[case] split columns of {SZI} x {szJ}", file=sys.stderr, flush=True)
    _need(torch, 150)
    lib, s, out = _bind(), _lib.stream_handle(), []
    for sz in (12, szJ):
        r = lambda lo, hi, seed, n=N, t=torch.float32: _rows(torch, sz, n, lo, hi, seed, t)
        A, Hz, B, Cc, W = r(-1, 1, 1), r(9, 11, 2), r(-1, 1, 3, N + 1), r(-1, 1, 4, N + 1), r(0, 1, 5, N + 1)
        for k in range(N + 1):
            W[k] += 10.0 * k          # z_w of the pressure gradient; omega writes it afterwards
        metric = r(0.9, 1.1, 7, 1, torch.float64)
        BC = torch.full((sz, SZI), -1, dtype=torch.int32, device="cuda")
        ctx = _ctx(torch, sz, N, metric)
        p = lambda *t: [x.data_ptr() for x in t]
        _lib.check(lib.sf_prsgrd(ctx, _lib.SF_FP32, *p(A, W, W, Hz), 9.8, 1025.0, *p(B, Cc), s), "sf_prsgrd")
        first = [_rows_of(x) for x in (B, Cc)]
        _lib.call("sf_set_maxflux_f32", ctx, *p(A, A, B, Cc, Hz), s)
        second = [_rows_of(x) for x in (B, Cc)]
        _lib.call("sf_omega_f32", ctx, *p(W, B, Cc, Hz, BC), s)
        third = [_rows_of(W)]
        new = torch.zeros_like(A[:1])
        one = _ctx(torch, sz, 1, metric)
        _lib.check(lib.sf_step3d_t(one, _lib.SF_FP32, *p(A, new, B, Cc, Hz[:1], Hz[1:]), 60.0, s), "sf_step3d_t")
        torch.cuda.synchronize()
        for c in (ctx, one):
            lib.sf_ctx_destroy(c)
        out.append(first + second + third + [_rows_of(new)])
        del A, Hz, B, Cc, W, metric, BC, new
        torch.cuda.empty_cache()
    names = ("prsgrd ru", "prsgrd rv", "Huon", "Hvom", "W", "tracer")
    bad = [(n, k) for n, a, b in zip(names, *out) for k in range(3) if not torch.equal(a[k], b[k])]
    assert not bad, bad
    assert all(o[3] for o in out[1]), [n for n, o in zip(names, out[1]) if not o[3]]


def _rows_of(t):
    """(first six rows, row six, last six rows, every row between equals row six)."""
    n, szJ = t.shape[0], t.shape[1]
    alike = all(bool((t[k, r:min(r + 2048, szJ - 6)] == t[k, 5]).all())
                for k in range(n) for r in range(6, szJ - 6, 2048))
    return t[:, :6].cpu(), t[:, 5].cpu(), t[:, -6:].cpu(), alike
