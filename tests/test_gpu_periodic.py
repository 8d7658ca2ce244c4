"""Pixels whose orbit becomes periodic are finished early by the persistent,
sliced and per-tile kernels: counts against the oracle where the comparisons
can go wrong.  Tolerance: none."""
import numpy as np
import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu

DEPTHS = (31, 33, 59, 61, 239, 241, 700, 3001)


def _check(ctx, oracle, rect, p, depth, w, h, fractal, path, julia=None):
    v = M.make_view(rect, precision=p, depth=depth, width=w, height=h, fractal=fractal, path=path,
                    family=M.FAMILY_JULIA if julia else M.FAMILY_MANDEL,
                    julia=julia or (None, None))
    ref = np.asarray(oracle.render(list(rect), precision=p, depth=depth, width=w, height=h,
                                   fractal=fractal, path=path, threads=16,
                                   family=1 if julia else 0,
                                   julia=julia or (None, None))).astype(np.int64)
    for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
        got = ctx.render_batch([(v, None, None)], mode=mode)[0][0]
        assert np.array_equal(got.astype(np.int64), ref), (p, depth, fractal, path, mode)
    with M.Server(ctx, slice_iters=101) as srv:
        got = srv.wait(srv.submit(v))[0]
    assert np.array_equal(got.astype(np.int64), ref), (p, depth, fractal, path, "server")


@pytest.mark.parametrize("depth", DEPTHS)
@pytest.mark.parametrize("path,p", [(M.PATH_DOUBLE, 64), (M.PATH_LD, 64), (M.PATH_MPFR, 24),
                                    (M.PATH_MPFR, 100), (M.PATH_MPFR, 256)])
def test_overviews_at_depths_around_the_comparisons(ctx, oracle, path, p, depth):
    """Cardioid and bulbs of every formula (the hybrid's cycles count the
    iteration's parity), their borders, and pixels that escape late."""
    rect = M.rect_from_center("-0.4", "0.1", "3.2", max(p, 64), 61, 43)
    for fractal in range(4):
        print(p, path, depth, fractal, flush=True)
        _check(ctx, oracle, rect, p, depth, 61, 43, fractal, path)


@pytest.mark.parametrize("path,p", [(M.PATH_DOUBLE, 64), (M.PATH_LD, 64), (M.PATH_MPFR, 128)])
def test_fixed_points_at_zero_and_on_the_axis(ctx, oracle, path, p):
    """c = 0 (orbits that square to nothing), c = -1 (0, -1, 0, ... exactly)
    and a real-axis frame whose middle row is exact."""
    for julia in (("0", "0"), ("-1", "0"), ("0.25", "0")):
        rect = M.rect_from_center("0", "0", "2", max(p, 64), 33, 21)
        print(p, path, julia, flush=True)
        _check(ctx, oracle, rect, p, 2000, 33, 21, 0, path, julia)


def test_queue_refills_forget_the_last_pixel(ctx, oracle):
    """More pixels than lanes, one block a CU: lanes go from periodic pixels to
    others in the middle of a launch."""
    for path, p in ((M.PATH_DOUBLE, 64), (M.PATH_MPFR, 64), (M.PATH_MPFR, 128)):
        kid = M.kernel_id(path, p)
        keep = ctx.tune_get(kid)[:2]
        try:
            ctx.tune_set(kid, blocks_per_cu=1, chunk=128)
            rect = M.rect_from_center("-0.75", "0", "3", 64, 480, 360)
            print(path, p, flush=True)
            _check(ctx, oracle, rect, p, 400, 480, 360, 0, path)
        finally:
            ctx.tune_set(kid, blocks_per_cu=keep[0], chunk=keep[1])
