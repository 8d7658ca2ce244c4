"""The wide RN arithmetic as the kernels compile it (29-bit-limb products,
rounding at a cut in the lowest words), on the CPU.  Tolerance: none."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_products_and_rounding_match_bit_by_bit(tmp_path):
    exe = tmp_path / "mp_wide_selftest"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe),
                    os.path.join(ROOT, "tests", "mp_wide_selftest.cpp")], check=True)
    for seed in (41, 42):
        r = subprocess.run([str(exe), str(seed), "20000"], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0 and r.stdout.startswith("0 mismatches"), r.stdout[-2000:]
        assert int(r.stdout.split(",")[1].split()[0]) > 0    # the exact path ran
