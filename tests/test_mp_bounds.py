"""Exponents of the RN arithmetic stay inside an int32, with zeros among the
operands: the host builds of the arithmetic, where a signed overflow ends the
program.  Tolerance: none."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("source, args", [("mp_zero_selftest", []),
                                          ("mp_fast_selftest", ["33", "2000"])])
def test_no_signed_overflow(tmp_path, source, args):
    exe = tmp_path / source
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=signed-integer-overflow",
                    "-fno-sanitize-recover=all", "-o", str(exe),
                    os.path.join(ROOT, "tests", source + ".cpp")], check=True)
    r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout + r.stderr)[-2000:]
    assert r.stdout.startswith("0 mismatches"), r.stdout[-2000:]
