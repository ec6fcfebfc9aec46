"""CPU checks of the packet walk's filters, compiled for the host with hipcc."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("name", ["open_filter_check", "relative_filter_check"])
def test_filter_never_rejects_a_leaf_within_the_bound(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.check_call([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "--cuda-host-only",
                           "-x", "hip", os.path.join(ROOT, "tests", "host", name + ".cpp"), "-o",
                           exe], stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
    assert "failures: 0" in out.stdout
