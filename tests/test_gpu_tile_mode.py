"""One launch a tile (BATCH_PER_TILE) iterates FP64 pixels as the persistent
launch does.  The orbits are bounded for their depth and slow to settle, so the
time is that of the iterations alone; the bound leaves the launches of four
tiles and the clock room (1.0 when this was written, 3.6 with the loop of a
branch a lane)."""
import numpy as np
import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu


def _view(fractal, w, h, depth, cx="-0.75", cy="0.0005", size="1e-6"):
    rect = M.rect_from_center(cx, cy, size, 64, w, h)
    return M.make_view(rect, precision=64, depth=depth, width=w, height=h, fractal=fractal,
                       path=M.PATH_DOUBLE)


def test_tiles_iterate_as_fast_as_the_queue(ctx):
    specs = [(_view(0, 640, 480, 3000), None, None)] * 4
    ms = {}
    for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
        ctx.render_batch(specs, mode=mode)
        ms[mode] = min(ctx.render_batch(specs, mode=mode)[1]["kernel_ms"] for _ in range(5))
    print(ms, flush=True)
    assert ms[M.BATCH_PER_TILE] < 1.35 * ms[M.BATCH_PERSISTENT]


@pytest.mark.parametrize("depth", [1, 2, 11, 12, 13, 59, 60, 61, 119, 121, 1000, 2**31 - 1])
def test_counts_at_the_edges_of_a_run(ctx, oracle, depth):
    """Depths about the exit tests and comparisons, partial waves, every formula."""
    for fractal in range(4):
        w, h = 37, 5
        # at the largest depth a view that every pixel leaves within a few iterations
        where = dict(cx="-0.5", cy="0.05", size="3") if depth <= 1000 else \
            dict(cx="1.5", cy="1.5", size="1")
        v = _view(fractal, w, h, depth, **where)
        ref = np.asarray(oracle.render([s.decode() for s in v._keep[:4]], precision=64,
                                       depth=min(depth, 1000), width=w, height=h, fractal=fractal,
                                       path=M.PATH_DOUBLE, threads=8)).astype(np.int64)
        assert depth <= 1000 or ref.all()
        got = ctx.render_batch([(v, None, None)], mode=M.BATCH_PER_TILE)[0][0]
        assert np.array_equal(got.astype(np.int64), ref), (depth, fractal)
