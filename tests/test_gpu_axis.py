"""Pixels on the real axis, whose wim is exactly zero in every iteration: counts
against the oracle (tolerance: none), and the time of a row on the axis against
the next one.  Both run to depth through nearly equal orbits; the bound leaves
room for the votes and the clock (1.8 to 2.2 when a zero was called rare and
every iteration done again)."""
import numpy as np
import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu


def _view(p, w, h, depth, fractal=0, julia=None, cx="-0.75", size="3", path=M.PATH_MPFR):
    rect = M.rect_from_center(cx, "0", size, p, w, h)
    return M.make_view(rect, precision=p, depth=depth, width=w, height=h, fractal=fractal,
                       family=M.FAMILY_JULIA if julia else M.FAMILY_MANDEL,
                       julia=julia or (None, None), path=path)


@pytest.mark.parametrize("p", [24, 64, 80, 128, 150, 192, 240, 256, 320])
def test_a_row_on_the_axis_takes_no_longer(ctx, p):
    # about a parabolic point: neither escaping nor periodic for thousands of iterations
    v = _view(p, 256, 256, 2000, size="1e-5" if p > 32 else "1e-3")

    def best(line):
        ctx.render(v, lines=(line, 1))
        return min(ctx.render(v, lines=(line, 1))[1]["kernel_ms"] for _ in range(6))

    a, b = best(128), best(127)
    print(p, a, b, flush=True)
    if not ctx.render(v, lines=(127, 2))[0].any() and p > 32:
        assert a < 1.3 * b


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
