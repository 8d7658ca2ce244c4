"""The per-operation probe times the loop that renders run: its iteration
against the time that a render of the same pixels takes for one more.  One
wave a SIMD, where the forms with and without votes lie furthest apart (2900
and 1700 cycles an iteration at 128 bits); the bound allows for the render's
refills and comparisons and for the clock."""
import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu


def test_probe_iterates_as_a_render_does(ctx):
    # orbits near a parabolic point: bounded for thousands of iterations, none periodic
    rect = M.rect_from_center("-0.75", "0.0005", "1e-6", 128, 640, 100)
    views = [M.make_view(rect, precision=128, depth=d, width=640, height=100) for d in (1000, 3000)]

    def best(f):
        f()
        return min(f() for _ in range(5))

    times = [best(lambda: ctx.render(v)[1]["kernel_ms"]) for v in views]
    assert not ctx.render(views[1])[0].any()
    render = (times[1] - times[0]) / 2000
    probe = (best(lambda: ctx.op_probe(views[0], 6, warm=500, reps=2000)) -
             best(lambda: ctx.op_probe(views[0], 0, warm=500, reps=2000))) / 2000
    print(f"render {render * 1e3:.4f} us, probe {probe * 1e3:.4f} us an iteration", flush=True)
    assert 0.75 < probe / render < 1.35
