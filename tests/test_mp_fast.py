"""The branch-light iteration of up to 8 words and of 10 whole ones (mdz_amd/csrc/mp_fast.h): on
the CPU against mp_rn.h, on the GPU against the oracle.  Tolerance: none."""
import os
import subprocess

import numpy as np
import pytest

import mdz_amd as M

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_iteration_matches_the_operations(tmp_path):
    exe = tmp_path / "mp_fast_selftest"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe),
                    os.path.join(ROOT, "tests", "mp_fast_selftest.cpp")], check=True)
    for seed in (31, 32):
        r = subprocess.run([str(exe), str(seed), "20000"], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0 and r.stdout.startswith("0 mismatches"), r.stdout[-2000:]


def _oracle(oracle, rect, p, depth, w, h, fractal):
    return np.asarray(oracle.render(list(rect), precision=p, depth=depth, width=w, height=h,
                                    fractal=fractal, path=M.PATH_MPFR, threads=8)).astype(np.int64)


@pytest.mark.gpu
@pytest.mark.parametrize("p", [2, 3, 20, 31, 32, 33, 63, 65, 95, 96, 97, 127, 161, 191, 225, 255])
def test_precisions_at_the_edges_of_a_word(ctx, oracle, p):
    """All bits cut from the lowest word but one, none, and few bits at all."""
    w, h = 35, 11
    for cx, cy, size, depth in (("0", "1", f"{2.0 ** -max(p - 16, 0):.9e}", p + 60),
                                ("-0.75", "0", "2.5", 300)):
        rect = M.rect_from_center(cx, cy, size, p, w, h)
        for fractal in range(4):
            v = M.make_view(rect, precision=p, depth=depth, width=w, height=h, fractal=fractal)
            print(p, cx, fractal, flush=True)
            ref = _oracle(oracle, rect, p, depth, w, h, fractal)
            for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
                got = ctx.render_batch([(v, None, None)], mode=mode)[0][0]
                assert np.array_equal(got.astype(np.int64), ref), (p, cx, fractal, mode)


@pytest.mark.gpu
def test_rows_on_the_real_axis_and_mixed_precisions_in_a_wave(ctx, oracle):
    """Tiles of few pixels share waves: their precisions (one class), formulas
    and distances from the real axis (on it, wim stays zero) differ by lane."""
    specs, refs = [], []
    for i, p in enumerate(list(range(225, 256)) + list(range(97, 128))):
        cy = ("0", "1e-30", "1e-9")[i % 3]
        w, h, depth = 5, 3, 200
        rect = M.rect_from_center("-1.9", cy, "0.01" if cy == "0" else "1e-20", p, w, h)
        v = M.make_view(rect, precision=p, depth=depth, width=w, height=h, fractal=i % 4)
        specs.append((v, None, None))
        refs.append(_oracle(oracle, rect, p, depth, w, h, i % 4))
    for mode in (M.BATCH_PERSISTENT, M.BATCH_PER_TILE):
        print("mode", mode, flush=True)
        for (v, _, _), got, ref in zip(specs, ctx.render_batch(specs, mode=mode)[0], refs):
            assert np.array_equal(got.astype(np.int64), ref), (v.precision, mode)
    with M.Server(ctx, slice_iters=13) as srv:
        ids = [srv.submit(v) for v, _, _ in specs]
        for i, ref in zip(ids, refs):
            assert np.array_equal(srv.wait(i)[0].astype(np.int64), ref)
