"""The Julia set of c = 0, where z squares itself away: exponents double every
iteration until a sum with the zero c flushes them.  The unit disk never
escapes at any precision and depth.  Tolerance: none."""
import numpy as np
import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [64, 128, 256, 320, 512, 1000, 1024])
def test_the_unit_disk_never_escapes(ctx, p):
    for w, h, depth in ((6, 5, 300), (256, 140, 100)):
        rect = M.rect_from_center("0", "0", "1", p, w, h)
        v = M.make_view(rect, precision=p, depth=depth, width=w, height=h,
                        family=M.FAMILY_JULIA, julia=("0", "0"))
        print(p, w, h, flush=True)
        for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
            assert not np.any(ctx.render_batch([(v, None, None)], mode=mode)[0][0]), (p, w, mode)
