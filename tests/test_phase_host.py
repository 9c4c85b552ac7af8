"""The fast variant's phase sine and cosine (phase_sincos, csrc/st_device.h),
built for the host by hipcc, against long double.  The reduced argument is
good to two roundings of pi/4 (2 * 5.6e-17), the series to its last two
operations (2 * 1.1e-16) and the product with r to one more: 4.5e-16 = 2 ulp
of 1.  No GPU is used.
"""
import os
import subprocess

import pytest

from conftest import ROOT

HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_phase_sincos(tmp_path):
    exe = str(tmp_path / "host_phase")
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-ffp-contract=off", "-w",
                    os.path.join(ROOT, "tests", "host_phase_main.cpp"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe, "4.5e-16"], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
