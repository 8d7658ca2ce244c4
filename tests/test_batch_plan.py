"""The launch plan of a batch (mdzg_plan_batch): four lanes a pixel and the class
whose pixels can take longest first while the batch leaves SIMDs idle; that class
first and spread over the CUs where the load is high and it does not fill the
chip itself; the order of kernel ids otherwise.  And batches of each kind against their tiles rendered alone.
Tolerance: none."""
import ctypes

import numpy as np
import pytest

import mdz_amd as M

NCU = 256


class _Tile(ctypes.Structure):
    _fields_ = [("kid", ctypes.c_int), ("depth", ctypes.c_longlong), ("pixels", ctypes.c_uint64)]


def _plan(tiles):
    arr = (_Tile * len(tiles))(*tiles)
    kids, how = (ctypes.c_int * 64)(), ctypes.c_int(-1)
    n = M.lib().mdzg_plan_batch(arr, len(tiles), NCU, kids, ctypes.byref(how))
    return list(kids[:n]), how.value


FOUR, SPREAD = 1, 2


def _k(p, path=M.PATH_MPFR):
    return M.kernel_id(path, p)


def _sheet(side=96):
    """A contact sheet: classes from FP64 to 1024 bits, the deepest, of side^2 pixels,
    the slowest.  Not made on import: the library must not load before torch, whose
    HIP runtime would be a second one in the process."""
    return [(0, 1000, 96 * 96), (_k(128), 2500, 64 * 64), (_k(64), 1000, 64 * 64),
            (_k(256), 2500, 96 * 96), (_k(256, M.PATH_GMP), 3000, 64 * 64),
            (_k(512), 1700, 64 * 64), (_k(320), 2000, 64 * 64), (_k(1024), 3600, side * side)]


# 28 tiles of 48x48 have a block a CU at most
@pytest.mark.parametrize("side, copies, how", [(96, 1, FOUR), (48, 28, SPREAD)])
def test_slowest_class_first_at_low_and_high_load(side, copies, how):
    tiles = _sheet(side)
    kids, got = _plan(tiles * copies)
    assert got == how
    assert kids[0] == _k(1024) and kids[-1] == 0
    assert sorted(kids) == sorted({t[0] for t in tiles})
    # 13.6M cycles at 512 bits, 6.9M at 256, 1.1M at 64
    assert kids.index(_k(512)) < kids.index(_k(256)) < kids.index(_k(64))


@pytest.mark.parametrize("side, copies", [(48, 29), (96, 30), (96, 32)])
def test_a_slowest_class_that_fills_the_chip_does_not_go_first(side, copies):
    tiles = _sheet(side) * copies
    # 65536 pixels are a block of one lane a pixel on each CU
    assert sum(t[2] for t in tiles if t[0] == _k(1024)) > 256 * NCU
    kids, how = _plan(tiles)
    assert how == 0 and kids == sorted(kids)


def test_many_classes_between_the_lines_go_by_id():
    nine = _sheet(48) + [(_k(700), 900, 64 * 64)]
    how = {}
    for copies in range(1, 29):
        kids, h = _plan(nine * copies)
        assert kids == sorted(kids) if h == 0 else kids[0] == _k(1024)
        how[copies] = h
    seen = list(how.values())
    assert seen == sorted(seen, key=[FOUR, 0, SPREAD].index) and set(seen) == {FOUR, 0, SPREAD}
    # up to eight classes have no such range
    assert {_plan(_sheet(48) * c)[1] for c in range(1, 29)} == {FOUR, SPREAD}


def test_order_is_by_time_not_by_id():
    # 320 bits have an id past the GMP buckets'
    kids, _ = _plan([(_k(1024), 100, 10), (_k(320), 100, 10), (_k(64), 100, 10)])
    assert kids == [_k(1024), _k(320), _k(64)] and kids != sorted(kids)


def test_a_class_alone_may_always_take_four_lanes():
    assert _plan([(_k(1024), 1000, 10**7)]) == ([_k(1024)], FOUR)


def _view(p, side, depth, path=M.PATH_MPFR, fractal=0):
    size = f"{2.0 ** -(p - 16):.17e}" if path == M.PATH_MPFR and p > 64 else "3"
    rect = M.rect_from_center("0", "1" if size != "3" else "0.1", size, p, side, side,
                              coords=path == M.PATH_GMP)
    return M.make_view(rect, precision=p, depth=depth, width=side, height=side, path=path,
                       fractal=fractal)


@pytest.mark.gpu
@pytest.mark.parametrize("nine, copies, how", [(False, 1, FOUR), (False, 8, FOUR), (True, 13, 0),
                                               (False, 27, SPREAD)])
def test_batches_of_each_plan(ctx, nine, copies, how):
    views = [_view(64, 48, 300, path=M.PATH_DOUBLE), _view(64, 32, 300, path=M.PATH_LD),
             _view(400, 40, 500), _view(512, 64, 600, fractal=2), _view(700, 33, 800),
             _view(256, 32, 300), _view(128, 32, 200, path=M.PATH_GMP), _view(1024, 48, 1100)]
    if nine:
        views += [_view(176, 32, 300)]
    assert _plan([(_k(v.precision, v.path), v.depth, v.real_width * v.real_height)
                  for v in views] * copies)[1] == how
    alone = [ctx.render(v)[0] for v in views]
    print(copies, flush=True)
    for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
        got = ctx.render_batch([(v, None, None) for v in views] * copies, mode=mode)[0]
        for i, g in enumerate(got):
            assert np.array_equal(g, alone[i % len(views)]), (i, mode)
