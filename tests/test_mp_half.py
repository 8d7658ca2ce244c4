"""The product that four lanes share, on the CPU, and which launches take that
form.  Tolerance: none."""
import ctypes
import os
import subprocess

import pytest

import mdz_amd as M

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_halves_join_to_the_product(tmp_path):
    exe = tmp_path / "mp_half_selftest"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe),
                    os.path.join(ROOT, "tests", "mp_half_selftest.cpp")], check=True)
    for seed in (51, 52):
        r = subprocess.run([str(exe), str(seed), "20000"], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0 and r.stdout.startswith("0 mismatches"), r.stdout[-2000:]


@pytest.mark.parametrize("p, four", [(256, False), (257, True), (319, True), (320, False),
                                     (321, True), (512, True), (1024, True)])
def test_which_launches_take_four_lanes(p, four):
    """Up to 128 pixels a CU from 10 words, but for 320 bits; never more."""
    kid = M.kernel_id(M.PATH_MPFR, p)
    pays = M.lib().mdzg_dev_quad_pays
    pays.argtypes = [ctypes.c_int, ctypes.c_uint64,
                     ctypes.c_int]
    assert [bool(pays(kid, n, 256)) for n in (1, 32768, 32769)] == [four, four, False]
    for path in (M.PATH_DOUBLE, M.PATH_GMP):
        assert not pays(M.kernel_id(path, 256), 1, 256)
