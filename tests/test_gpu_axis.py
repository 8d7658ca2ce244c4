"""Pixels on the real axis, whose wim is exactly zero in every iteration, which the
branch-light loop calls rare and does again: counts against the oracle
(tolerance: none)."""
import numpy as np
import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu


def _view(p, w, h, depth, fractal=0, julia=None, cx="-0.75", size="3", path=M.PATH_MPFR):
    rect = M.rect_from_center(cx, "0", size, p, w, h)
    return M.make_view(rect, precision=p, depth=depth, width=w, height=h, fractal=fractal,
                       family=M.FAMILY_JULIA if julia else M.FAMILY_MANDEL,
                       julia=julia or (None, None), path=path)


@pytest.mark.parametrize("p", [24, 64, 80, 128, 150, 192, 200, 256, 320])
def test_counts_on_the_axis(ctx, oracle, p):
    """Square frames about 0: a row lies on the axis; every formula, and Julia sets of a real c."""
    w, h, depth = 32, 32, 300
    lines = (14, 5)
    for fractal in range(4):
        for julia in (None, ("-1", "0"), ("-0.75", "0"), ("0", "0"), ("0.25", "0")):
            v = _view(p, w, h, depth, fractal, julia, cx="0" if julia else "-0.75", size="4")
            ref = np.asarray(oracle.render([s.decode() for s in v._keep[:4]], precision=p,
                                           depth=depth, width=w, height=h, fractal=fractal,
                                           path=M.PATH_MPFR, threads=8, lines=(*lines, 1),
                                           family=1 if julia else 0,
                                           julia=julia or (None, None))).astype(np.int64)
            for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
                got = ctx.render_batch([(v, lines, None)], mode=mode)[0][0]
                assert np.array_equal(got.astype(np.int64), ref), (p, fractal, julia, mode)
            with M.Server(ctx, slice_iters=7) as srv:
                got = srv.wait(srv.submit(v, lines=lines))[0]
                assert np.array_equal(got.astype(np.int64), ref), (p, fractal, julia)


def test_long_stays_on_the_axis(ctx):
    """Many runs on: the exponent of a zero does not creep up on the other values."""
    a, b = (_view(128, 256, 256, d, size="1e-5") for d in (200000, 2000))
    got = ctx.render(a, lines=(128, 1), cols=(0, 128))[0]
    assert np.array_equal(got, ctx.render(b, lines=(128, 1), cols=(0, 128))[0]) and not got.any()
