"""Four lanes a pixel (k_quad.h): launches at both sides of the rule, partial
waves and quads, queues that refill, every formula, deep and on the axis,
against the oracle; and slices that go from one form to the other.
Tolerance: none."""
import numpy as np
import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu


def _ref(oracle, rect, p, depth, w, h, fractal, julia=None):
    return np.asarray(oracle.render(list(rect), precision=p, depth=depth, width=w, height=h,
                                    fractal=fractal, path=M.PATH_MPFR, threads=16,
                                    family=1 if julia else 0,
                                    julia=julia or (None, None))).astype(np.int64)


def _view(p, w, h, depth, fractal, cx="0", cy="1", size=None, julia=None):
    size = size or f"{2.0 ** -(min(p, 1000) - 16):.17e}"
    rect = M.rect_from_center(cx, cy, size, p, w, h)
    return rect, M.make_view(rect, precision=p, depth=depth, width=w, height=h, fractal=fractal,
                             family=M.FAMILY_JULIA if julia else M.FAMILY_MANDEL,
                             julia=julia or (None, None))


@pytest.mark.parametrize("p", [257, 320, 350, 384, 448, 500, 512, 640, 700, 768, 896, 1000, 1024])
def test_small_tiles(ctx, oracle, p):
    for w, h, fractal, kw in ((1, 1, 0, {}), (17, 1, 1, {}), (5, 13, 2, {}), (9, 9, 3, {}),
                              (11, 7, 0, dict(cx="-1.9", cy="0", size="0.5")),
                              (11, 7, 2, dict(cx="-0.5", cy="0", size="3")),
                              (6, 5, 0, dict(cx="-1", julia=("0", "1"))),
                              (6, 5, 0, dict(cx="0", cy="0", size="1", julia=("0", "0")))):
        rect, v = _view(p, w, h, p + 50, fractal, **kw)
        print(p, w, h, fractal, kw, flush=True)
        got = ctx.render(v)[0]
        assert np.array_equal(got.astype(np.int64),
                              _ref(oracle, rect, p, p + 50, w, h, fractal, kw.get("julia")))


def test_both_sides_of_the_rule_agree(ctx):
    """The same view as one launch past the rule and as bands below it."""
    for p in (320, 500, 1024):
        _, v = _view(p, 256, 160, 400, 0, size="1e-60")
        whole = ctx.render(v)[0]
        print(p, flush=True)
        for line0, n in ((0, 128), (128, 32)):
            part = ctx.render(v, lines=(line0, n))[0]
            assert np.array_equal(part, whole[line0:line0 + n]), (p, line0)


def test_slices_change_form_and_mix_precisions(ctx, oracle):
    """Requests of one class joining and leaving move the class across the
    rule between slices; the saved state serves both forms."""
    rect, small = _view(500, 24, 16, 700, 0)
    ref = _ref(oracle, rect, 500, 700, 24, 16, 0)
    _, other = _view(460, 20, 12, 300, 2)
    _, big = _view(500, 256, 144, 120, 0, cx="-0.1", cy="0.2", size="1e-9")
    alone = {id(v): ctx.render(v)[0] for v in (other, big)}
    with M.Server(ctx, slice_iters=23) as srv:
        first = srv.submit(small)
        rest = [(v, srv.submit(v)) for v in (big, other, big)]
        assert np.array_equal(srv.wait(first)[0].astype(np.int64), ref)
        for v, i in rest:
            assert np.array_equal(srv.wait(i)[0], alone[id(v)])


def test_depth_at_the_limit_of_int32(ctx):
    """A pixel that escapes long before the largest depth there is."""
    _, v = _view(400, 3, 2, 2**31 - 1, 0)
    _, w = _view(400, 3, 2, 5000, 0)
    assert np.array_equal(ctx.render(v)[0], ctx.render(w)[0])
