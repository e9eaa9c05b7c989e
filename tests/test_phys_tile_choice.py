"""sf_phys_fused_tile (host only): the tile of a fused physics substep on both sides of every
line of its rule."""
from __future__ import annotations

import ctypes as C

import pytest

from sailfish_amd import _lib
from sailfish_amd.phys2d import _bind

PLAIN, COUPLED, CLOSURE = 0, 1, 2


def _tile(prec, form, szI, szJ):
    a, b = C.c_int32(), C.c_int32()
    _lib.check(_bind().sf_phys_fused_tile(prec, form, szI, szJ, C.byref(a), C.byref(b)), "sf_phys_fused_tile")
    return a.value, b.value


@pytest.mark.parametrize("szI,szJ,f64,f32", [
    (256, 128, (16, 8), (16, 8)),       # 256 16 x 8 tiles
    (257, 128, (32, 8), (32, 8)),       # 272
    (352, 184, (32, 8), (32, 8)),       # 253 32 x 8 tiles, no bands
    (416, 160, (64, 8), (32, 8)),       # 260, no bands
    (512, 144, (32, 8), (32, 8)),       # 288
    (480, 248, (64, 8), (64, 8)),       # 465, no bands; 248 64 x 8
    (544, 240, (64, 4), (32, 8)),       # 510, no bands; 270 64 x 8, 540 64 x 4
    (512, 256, (32, 8), (32, 8)),       # 512
    (544, 256, (64, 4), (32, 8)),       # 544; 288 64 x 8, 576 64 x 4
    (513, 255, (64, 4), (32, 8)),
    (672, 248, (64, 4), (64, 8)),       # 651, no bands; 682 64 x 4
    (768, 256, (64, 4), (32, 8)),       # 768; 768 64 x 4
    (640, 320, (64, 8), (64, 8)),       # 800; 800 64 x 4
    (2048, 1024, (64, 8), (64, 8)),
])
def test_plain(szI, szJ, f64, f32):
    assert _tile(_lib.SF_FP64, PLAIN, szI, szJ) == f64 and _tile(_lib.SF_FP32, PLAIN, szI, szJ) == f32


@pytest.mark.parametrize("szI,szJ,f64,f32", [
    (128, 64, (16, 8), (16, 8)),
    (640, 184, (32, 8), (32, 8)),       # 460, no bands
    (480, 248, (32, 8), (64, 4)),       # 465, no bands; 496 64 x 4
    (512, 256, (32, 8), (32, 8)),
    (544, 256, (32, 8), (64, 4)),
    (640, 296, (64, 8), (64, 4)),       # 740, no bands
    (768, 384, (32, 8), (64, 4)),       # 1152, 576 64 x 8
    (832, 344, (32, 8), (64, 4)),       # 1118, no bands; 559 64 x 8
    (1024, 512, (64, 8), (64, 8)),      # 1024 64 x 8
])
def test_coupled(szI, szJ, f64, f32):
    assert _tile(_lib.SF_FP64, COUPLED, szI, szJ) == f64 and _tile(_lib.SF_FP32, COUPLED, szI, szJ) == f32


def test_closure_and_refusals():
    for prec in (_lib.SF_FP64, _lib.SF_FP32):
        assert _tile(prec, CLOSURE, 512, 128) == (32, 8) and _tile(prec, CLOSURE, 513, 128) == (64, 4)
    for args in ((_lib.SF_FP64, 3, 64, 64), (_lib.SF_FP64, -1, 64, 64), (7, 0, 64, 64), (_lib.SF_FP64, 0, 3, 64)):
        with pytest.raises(_lib.SailfishError):
            _tile(*args)
