"""CPU check of the range walk's float32 filter, compiled for the host with hipcc."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_sure_pairs_are_sure(tmp_path):
    exe = str(tmp_path / "range_filter_check")
    subprocess.check_call([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "--cuda-host-only",
                           "-x", "hip",
                           os.path.join(ROOT, "tests", "host", "range_filter_check.cpp"), "-o",
                           exe], stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
    assert "failures: 0" in out.stdout
