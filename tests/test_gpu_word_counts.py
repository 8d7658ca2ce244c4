"""The RN kernels at the smallest and largest precision of the word counts
between the powers of two (5, 7, 10, 14, 20 and 28 words), against the
oracle.  Tolerance: none (counts are whole numbers)."""
import numpy as np
import pytest

import mdz_amd as M

W, H = 33, 9


def _words(p):
    return next(n for n in (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32) if 32 * n >= p)


EDGES = [129, 159, 160, 193, 224, 257, 288, 289, 320, 385, 416, 448, 513, 544, 577, 640,
         769, 800, 833, 896]


def _view(p, fractal, julia):
    """Around the Misiurewicz point c = i (or the Julia set of it around its
    repelling point -1 + i), as deep as p allows, where escape counts vary
    from pixel to pixel."""
    width = f"{2.0 ** -(min(p, 1000) - 16):.17e}"
    rect = M.rect_from_center("-1" if julia else "0", "1", width, p, W, H)
    return rect, M.make_view(rect, precision=p, depth=p + 60, width=W, height=H, fractal=fractal,
                             family=M.FAMILY_JULIA if julia else M.FAMILY_MANDEL,
                             julia=("0", "1") if julia else (None, None))


def test_kernel_ids_of_saved_tables_stay():
    """A saved table's rows name kernels by id: every word count (and GMP
    bucket) that had an id keeps it, and no two kernels share one."""
    old = {1: 1, 2: 3, 3: 5, 4: 7, 6: 9, 8: 11, 12: 13, 16: 15, 24: 17, 32: 19}
    for n, kid in old.items():
        assert M.kernel_id(M.PATH_MPFR, 32 * n) == kid + 1
        assert M.kernel_id(M.PATH_MPFR, 32 * n - 1) == kid
    assert [M.kernel_id(M.PATH_GMP, p) for p in (128, 256, 512, 1024)] == [21, 22, 23, 24]
    ids = {}
    for p in range(2, 1025):
        ids.setdefault(M.kernel_id(M.PATH_MPFR, p), set()).add((_words(p), 32 * _words(p) == p))
    assert len(ids) == 32 and all(len(v) == 1 for v in ids.values())


@pytest.mark.gpu
@pytest.mark.parametrize("p", EDGES)
def test_counts_at_the_edges_of_word_counts(ctx, oracle, p):
    for fractal, julia in ((0, False), (0, True), (1, False), (2, False), (3, False)):
        rect, v = _view(p, fractal, julia)
        print(p, fractal, julia, flush=True)
        ref = oracle.render(list(rect), precision=p, depth=p + 60, width=W, height=H,
                            fractal=fractal, path=M.PATH_MPFR, threads=8,
                            family=1 if julia else 0,
                            julia=("0", "1") if julia else (None, None))
        ref = np.asarray(ref).astype(np.int64)
        for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
            got = ctx.render_batch([(v, None, None)], mode=mode)[0][0]
            assert np.array_equal(got.astype(np.int64), ref), (p, fractal, julia, mode)
        with M.Server(ctx, slice_iters=37) as srv:
            got, _ = srv.wait(srv.submit(v))
        assert np.array_equal(got.astype(np.int64), ref), (p, fractal, julia, "server")
