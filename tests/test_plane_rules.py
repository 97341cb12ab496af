"""The rules that choose a plane stage and a queue order, asked of the built
library (they need no device).

* Beside a chain of Kleinman-Bylander products, the stage per wave is not taken
  where the filter step was measured slower with it: 128^3 up to 32 orbitals
  (FP64, 8 orbitals: 844 us against 574), 48^3 in FP64, 64^3 in FP32; and the
  chain is not put ahead of a workgroup-wide stage whose pair grids reach 320
  MiB (64^3, FP32, from 320 orbitals), nor at 192^3 or in the split form.
* The largest sphere at 128^3 whose planes fit LDS in the stage per wave: |k| <=
  23 in FP64 (160 KB hold 47 rows), every pruned one (|k| <= 31) in FP32.
"""
import ctypes
import os

import pytest

from sdft_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.lib_path()), reason="library not built")

FP64, FP32 = 0, 1


@pytest.fixture(scope="module")
def lib():
    lib = ctypes.CDLL(build.lib_path())
    b, i = ctypes.c_bool, ctypes.c_int
    f = lib._ZN4sdft14wave_beside_kbEiii
    f.restype, f.argtypes = b, [i, i, i]
    g = lib._ZN4sdft14kb_chain_firstEiiibb
    g.restype, g.argtypes = b, [i, i, i, b, b]
    h = lib._ZN4sdft14wplane_lds_forEiii
    h.restype, h.argtypes = ctypes.c_size_t, [i, i, i]
    return f, g, h


def test_stage_beside_products(lib):
    wave = lib[0]
    for prec in (FP64, FP32):
        for npairs in (1, 2, 4, 15, 16):
            assert not wave(128, prec, npairs)
        for npairs in (17, 20, 32, 64):
            assert wave(128, prec, npairs)
        for npairs in (1, 16, 17, 128):
            assert wave(96, prec, npairs)
            assert wave(48, prec, npairs) == (prec == FP32)
            assert wave(64, prec, npairs) == (prec == FP64)


def test_order_of_products(lib):
    first = lib[1]
    for n, prec, at in ((64, FP32, 160), (48, FP64, 190), (128, FP64, 10)):
        assert first(n, prec, at - 1, False, False)
        assert not first(n, prec, at, False, False)
        assert first(n, prec, at, True, False)
        assert not first(n, prec, 1, False, True)
    for prec in (FP64, FP32):
        assert not first(192, prec, 1, False, False)


def test_lds_limit_of_the_stage_per_wave(lib):
    lds = lib[2]
    assert 0 < lds(128, FP64, 2 * 23 + 1) <= 160 * 1024
    assert lds(128, FP64, 2 * 24 + 1) == 0
    assert 0 < lds(128, FP32, 2 * 31 + 1) <= 160 * 1024
    for n in (24, 32, 36, 48, 64, 96):
        for prec in (FP64, FP32):
            assert 0 < lds(n, prec, 2 * ((n - 1) // 4) + 1) <= 160 * 1024
