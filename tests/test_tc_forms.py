"""How condensed products with a plan are launched, on either side of each line that was measured (no GPU needed)."""
import ctypes

import pytest

from helpers import tc_form


@pytest.mark.parametrize("t,mb,feat,groups,out,form", [
    # 32-row tiles of a few steps, a last unit of 32 or 64 features: one step on its way, so that three wavefronts fit a SIMD
    (32, 1875, 160, 10, "f16", "128 by 4, one step"),
    (32, 1875, 192, 16, "f32", "128 by 4, one step"),
    (32, 5292, 160, 9, "f32", "128 by 2, one step"),
    (32, 5292, 192, 9, "f16", "128 by 2, one step"),
    (32, 5292, 192, 11, "f16", "128 by 2"),
    (32, 5292, 256, 9, "f16", "128 by 2"),
    (32, 625, 128, 8, "f16", "128 by 4"),
    (32, 1400, 128, 8, "f16", "128 by 4, one step"),
    # 16 rows: a little sooner with fp32 results
    (16, 10584, 160, 5, "f32", "128 by 2, one step"),
    (16, 10584, 160, 5, "f16", "128 by 2"),
    (16, 10584, 192, 4, "f16", "128 by 2, one step"),
    (16, 10584, 192, 8, "f32", "128 by 2"),
    (16, 10584, 224, 5, "f32", "128 by 2"),
    (16, 3125, 128, 20, "f32", "128 by 4"),
    # 8 rows: two units of 64 for 128 features of tiles of several steps
    (8, 21168, 128, 13, "f16", "64 by 2"),
    (8, 6250, 128, 9, "f32", "64 by 2"),
    (8, 21168, 128, 8, "f32", "128 by 2, one step"),
    (8, 4125, 128, 12, "f32", "128 by 4, one step"),
    (8, 21168, 128, 3, "f16", "128 by 2, one step"),
    (8, 21168, 256, 13, "f16", "128 by 2, one step"),
    (8, 2500, 224, 3, "f32", "128 by 2"),
    (8, 4125, 192, 4, "f16", "128 by 2"),
    # 32 features in a unit of their own; not in a small launch of 32-row tiles or a turn of 8-row ones
    (8, 1793, 160, 13, "f16", "64 by 4"),
    (8, 1250, 160, 13, "f16", "128 by 4, one step"),
    (8, 2050, 160, 3, "f16", "128 by 4, one step"),
    (16, 1250, 160, 5, "f16", "128 by 4"),
    (8, 2500, 160, 3, "f32", "128 by 2"),
    (32, 375, 160, 8, "f32", "64 by 4"),
    (32, 1032, 160, 10, "f32", "128 by 4, one step"),
    # up to 64 features
    (16, 1250, 64, 5, "f16", "64 by 4"),
    (16, 10584, 32, 3, "f16", "32 by 2"),
])
def test_form(t, mb, feat, groups, out, form):
    assert tc_form(t, out, mb, feat, groups * mb) == form


@pytest.mark.parametrize("t,out,mb,feat,nnzb,pieces", [(12, 0, 4, 64, 4, 0), (16, 1, 4, 64, 4, 0), (16, 0, 0, 64, 0, 0),
                                                       (16, 0, 4, 0, 4, 0), (16, 0, 4, 64, -1, 0), (16, 0, 4, 64, 4, -1)])
def test_what_no_product_is(t, out, mb, feat, nnzb, pieces):
    from sparsetir_amd import _lib

    assert _lib.lib().stir_tc_form(t, out, mb, feat, ctypes.c_int64(nnzb), ctypes.c_int64(pieces)) == -1
