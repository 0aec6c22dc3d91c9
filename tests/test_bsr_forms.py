"""How BSR products are launched, on either side of each line that was measured (256 compute units; no GPU needed)."""
import ctypes
import random

import pytest

from helpers import bsr_form


@pytest.mark.parametrize("mb,nb,blk,steps,feat,form", [
    # 32-row slices: order of length by the steps, the X of a tile and how many wavefronts there are
    (2048, 512, 32, 10, 1024, "128 by 1"),
    (2048, 512, 32, 16, 1024, "256 by 1 ranked"),
    (2048, 512, 32, 16, 256, "128 by 1"),           # one feature tile
    (2048, 512, 32, 32, 256, "256 by 1 ranked"),
    (2048, 207, 32, 16, 1024, "256 by 1"),          # X in an L2
    (2048, 207, 32, 32, 1024, "256 by 1 ranked"),
    (250, 512, 32, 16, 1024, "128 by 1"),           # few
    (2048, 512, 32, 16, 544, "128 by 1"),           # a last tile mostly empty
    (512, 512, 32, 51, 4096, "256 by 1 ranked"),
    (400, 170, 96, 6, 512, "LDS 32 x 128"),
    (400, 170, 96, 16, 512, "256 by 1 ranked"),
    (1300, 325, 96, 8, 1504, "LDS 32 x 256"),
    # steps in turn, by the tiles a compute unit has
    (291, 58, 32, 4, 160, "128 by 2"),
    (107, 48, 32, 5, 544, "128 by 2"),
    (107, 48, 32, 9, 544, "128 by 4"),
    (256, 66, 32, 5, 512, "128 by 2"),
    (258, 66, 32, 5, 512, "128 by 1"),
    (37, 441, 32, 102, 2848, "128 by 1"),            # far more X than the L2s hold
    (57, 18, 96, 8, 704, "128 by 1"),
    (18, 12, 128, 3, 1344, "LDS 64 x 128"),          # few steps: 64 rows by a workgroup
    (77, 115, 128, 21, 64, "LDS 64 by 8"),
    (22, 126, 128, 136, 864, "128 by 4"),            # 2.4 tiles a compute unit
    (22, 126, 128, 47, 864, "128 by 2"),
    (26, 126, 128, 136, 864, "LDS 64 x 128"),        # 2.8
    (102, 140, 64, 21, 416, "128 by 2"),             # 3.2
    (102, 14, 64, 21, 416, "LDS 64 x 128"),          # little X
    (51, 7, 128, 21, 416, "LDS 64 x 128 by rows"),
    (17, 150, 96, 275, 224, "LDS 64 by 8"),          # 64 features by eight: a turn of them
    (17, 150, 96, 99, 224, "128 by 8"),              # ... of which the last are half empty
    (30, 150, 96, 275, 96, "LDS 64 by 8"),
    (40, 150, 96, 275, 96, "128 by 8"),              # ... of one tile of 128
    (360, 190, 64, 234, 64, "LDS 64 by 8"),          # two turns of 64 features alone
    (360, 190, 64, 31, 64, "128 by 2"),
    # 64 rows by four wavefronts
    (1024, 256, 64, 12, 1024, "LDS 64 x 256"),
    (1024, 256, 64, 24, 1024, "LDS 64 x 256 ranked"),
    (256, 256, 64, 16, 256, "LDS 64 x 128"),
    (128, 128, 128, 51, 4096, "LDS 64 x 256 ranked by rows"),
    (12, 40, 128, 30, 3008, "LDS 64 x 128"),
    (45, 45, 128, 20, 1024, "LDS 64 x 128 by rows"),
    # 16-row slices
    (4096, 1025, 16, 10, 1024, "128 by 1"),
    (4096, 1025, 16, 18, 1024, "256 by 1 ranked"),
    (1024, 420, 16, 10, 512, "256 by 1"),
    (521, 872, 16, 32, 3168, "128 by 1 ranked"),      # far more X than an L2 holds, many tiles
    (521, 872, 16, 44, 3168, "256 by 1 ranked"),
    (521, 700, 16, 32, 3168, "256 by 1 ranked"),
    (1024, 872, 16, 32, 1024, "256 by 1 ranked"),     # few
    (100, 902, 16, 18, 2912, "128 by 1, one step"),   # a turn of wavefronts over far more X than the L2s hold
    (79, 657, 16, 20, 3616, "128 by 1, one step"),
    (44, 626, 16, 26, 4064, "128 by 1"),
    (44, 626, 16, 14, 4064, "128 by 4"),
    (79, 600, 16, 20, 3616, "128 by 4"),
    (250, 657, 16, 20, 992, "128 by 4"),              # few feature tiles
    (1100, 341, 48, 10, 1024, "128 by 2, two tiles"),
    (137, 84, 80, 27, 1824, "256 by 4"),
    (137, 84, 80, 29, 1824, "256 by 4 ranked"),
    (330, 320, 48, 39, 1280, "256 by 4 ranked"),
    (763, 273, 48, 30, 256, "128 by 4"),              # one feature tile
    (763, 273, 48, 36, 480, "256 by 4 ranked"),
    (763, 371, 48, 30, 480, "256 by 4 ranked"),       # far more X than an L2 holds
    (137, 84, 80, 29, 256, "128 by 4"),
    (137, 84, 80, 29, 1312, "128 by 4"),              # a last tile of 256 mostly empty
    (137, 84, 80, 35, 1312, "128 by 4"),
    (137, 84, 80, 36, 1312, "128 by 1 ranked"),
    (78, 108, 112, 26, 832, "128 by 4"),
    (430, 650, 48, 15, 608, "128 by 2, two tiles"),   # far more X than an L2 holds
    (430, 650, 48, 17, 608, "128 by 4"),
    (269, 331, 48, 25, 1248, "128 by 4"),             # blocks of 48 with much X
    (269, 120, 48, 25, 1248, "256 by 4"),
    (30, 84, 80, 29, 1824, "128 by 4"),               # few
    (97, 38, 112, 27, 2720, "256 by 4"),              # X in an L2
    (97, 38, 112, 15, 2720, "128 by 2, two tiles"),
    (97, 38, 112, 4, 2720, "128 by 1"),
    (328, 190, 48, 29, 1376, "128 by 4"),
    (224, 336, 48, 29, 2208, "128 by 4"),
    (97, 38, 112, 19, 2400, "128 by 2, two tiles"),   # an odd number of tiles of 128
    (22, 174, 48, 11, 320, "128 by 4"),
    (600, 650, 48, 7, 256, "128 by 2, two tiles"),
    (3693, 559, 48, 11, 320, "128 by 1"),
    (1214, 659, 80, 10, 416, "128 by 2, two tiles"),
    (3, 68, 144, 196, 416, "LDS 64 by 8"),            # long rows, much X, a turn of 64 features by eight
    (3, 68, 144, 99, 416, "128 by 8"),
    (3, 50, 144, 196, 416, "128 by 8"),
    (3000, 68, 80, 8, 800, "128 by 1"),
    (3000, 68, 80, 20, 800, "256 by 4"),            # A beyond the last level
])
def test_form(mb, nb, blk, steps, feat, form):
    nnzb = -(-steps * mb * 32 // blk)
    assert bsr_form(mb, nb, blk, feat, nnzb) == form


@pytest.mark.parametrize("mb,nb,blk,steps,feat,form,floats", [
    # several wavefronts to a tile store fp32 results sooner
    (62, 35, 32, 2, 2048, "128 by 1", "128 by 2"),
    (199, 36, 32, 2, 352, "128 by 1", "128 by 2"),
    (38, 13, 96, 2, 608, "128 by 1", "128 by 2"),
])
def test_form_with_few_steps(mb, nb, blk, steps, feat, form, floats):
    nnzb = -(-steps * mb * 32 // blk)
    assert bsr_form(mb, nb, blk, feat, nnzb) == form and bsr_form(mb, nb, blk, feat, nnzb, floats=True) == floats


def test_16_row_slices_name_instances_that_exist():
    """Tiles of 256 features are by one wavefront in blocks of 16 and by four in others; one step on its way in blocks of 16 only."""
    rng = random.Random(3)
    for _ in range(20000):
        blk = rng.choice([16, 48, 80, 112, 144])
        mb, nb, feat = (int(2 ** rng.uniform(0, top)) for top in (12, 11, 7))
        form = bsr_form(mb, nb, blk, 32 * feat, int(mb * nb * 2 ** rng.uniform(-8, 0)), floats=rng.random() < 0.5)
        if form.startswith("256"):
            assert form.startswith("256 by 1" if blk == 16 else "256 by 4")
        assert blk == 16 or "one step" not in form


def test_sizes_whose_offsets_do_not_fit():
    """Where a load's offset from the wavefront's first may not fit 32 bits: kernels that allow for more."""
    assert bsr_form(4, 4, 32, 1 << 25, 16) == "LDS 32 x 256"
    assert bsr_form(64, 4, 4096 + 32, 4096, 64) == "LDS 32 x 256"
    assert bsr_form(64, 4, 4096 + 16, 4096, 64) == "128 by 2, two tiles"
    assert bsr_form(64, 4, 32768 + 16, 4096, 64) == "LDS 64 by 8"
    assert bsr_form(4, 4, 16, 1 << 27, 16) == "LDS 64 by 8"


@pytest.mark.parametrize("mb,nb,blk,feat,nnzb,cus", [(0, 4, 32, 64, 0, 256), (4, 4, 24, 64, 4, 256), (4, 4, 32, 0, 4, 256),
                                                     (4, 4, 32, 64, -1, 256), (4, 4, 32, 64, 4, 0)])
def test_what_no_product_is(mb, nb, blk, feat, nnzb, cus):
    from sparsetir_amd import _lib

    assert _lib.lib().stir_bsr_form(cus, mb, nb, blk, feat, ctypes.c_int64(nnzb), 0) == -1
