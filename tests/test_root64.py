"""The FP64 kernels' square roots and quotients without range handling, on the
host: equal to the IEEE operations over the range declared for them, from seeds
worse than the hardware's (its reciprocal square root is within 2^-24.1 over
[1, 4); here 2^-23), with a reciprocal of the root good to 1.25 ulp, which is
what the quotients' bound rests on."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_roots_and_quotients(tmp_path):
    exe = str(tmp_path / "root64_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "root64_check.cpp")],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([exe, "2000000"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
