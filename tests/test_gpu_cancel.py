"""A cancelled job ends within a bounded number of iterations, or one chunk where
that is longer, whatever the chunk: there were 16 chunks to a look at the flag.
The chunks here made that 76 to 130 ms against 10 to 17; the bound is 40."""
import time

import pytest

import mdz_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p, side, chunk", [(64, 512, 4096), (128, 512, 4096), (400, 64, 4096),
                                            (512, 256, 2048), (1024, 256, 1024)])
def test_long_chunks_do_not_hold_a_cancelled_job(p, side, chunk):
    # bounded for far more than the depth, and never periodic
    rect = M.rect_from_center("-0.75", "1e-9", "1e-12", p, side, side)
    v = M.make_view(rect, precision=p, depth=400000, width=side, height=side)
    # a context of its own: its first job and the cancel flag's copy lie on two hardware queues
    with M.Context(0) as ctx:
        ctx.tune_set(M.kernel_id(M.PATH_MPFR, p), chunk=chunk)
        print(p, flush=True)
        job = ctx.submit([(v, None, None)])
        time.sleep(0.01)
        t = time.perf_counter()
        job.cancel()
        rc = job.wait()[0]
        t = time.perf_counter() - t
        job.free()
    print(f"{p} bits: {t * 1e3:.1f} ms after the cancel", flush=True)
    assert rc == -4 and t < 0.04
